"""Timed cases: what a user of this engine has it do, through its public entry points.

A case is a dict of plain values; its ``kind`` says which entry points it goes
through:

icd      a restarted reconstruction on the stepwise API (``Icd.upload``,
         ``iterate``, ``download``), as each stage of a multi-resolution run does:
         the starting volume and ring offsets go in, the iterated ones come back.
         Options: frames (4D), voxels of several bins (the coarse stages), edge-only
         updates, phase contrast.
batch    several slabs of different sizes advanced together by ``IcdBatch``.
fbp      the filtered-backprojection start alone.
infer    the warm-start network on a volume in device memory (``xt_unet_forward``).
train    its loss and gradient (``xt_unet_loss_grad``).
offset   the allocation-free ring-offset update on device arrays.

The scans are ellipsoids whose line integrals are taken in closed form, with
Poisson counts, zingers and ring offsets, made on the GPU from the seed alone.
The lines in flight and the workgroup width are pinned, as in a program that wants
one schedule from run to run (left alone, the create-time autotuner picks them from
a timing): the width and the number that the autotuner settles on for such sizes.
"""
import ctypes
import dataclasses
import importlib.util
import math
import os
import shutil
import sys
import tempfile

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "timbir-python_amd")


def _load():
    if "timbir_python_amd" not in sys.modules:
        spec = importlib.util.spec_from_file_location(
            "timbir_python_amd", os.path.join(_PKG, "__init__.py"),
            submodule_search_locations=[_PKG])
        sys.modules["timbir_python_amd"] = mod = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(mod)
    from timbir_python_amd import synth, xt_hip
    return synth, xt_hip


synth, xt_hip = _load()
WEIGHTS = os.path.join(_PKG, "weights", "unet_warmstart_256x256x16.npz")

# (level, C_in, C_out) of the network's 3x3x3 convolutions, in parameter order
CONVS = [(0, 1, 16), (0, 16, 16), (1, 16, 32), (1, 32, 32), (2, 32, 64), (2, 64, 64),
         (3, 64, 128), (3, 128, 128), (2, 192, 64), (2, 64, 64), (1, 96, 32), (1, 32, 32),
         (0, 48, 16), (0, 16, 16)]


# -- the cases --------------------------------------------------------------
def listed():
    return [
        # the production slab (512^2 x 32, 1024 views) in the final stage of a
        # multi-resolution run: two iterations with the FP64 recompute of e, the
        # benchmark's iteration
        dict(name="slab", kind="icd", N=512, Nz=32, views=1024, threads=256, omp=32, iters=2,
             resync=1),
        # the small plain 3D slab (128^2 x 8, 256 views): launches and latencies count
        dict(name="small", kind="icd", N=128, Nz=8, views=256, threads=256, omp=4, iters=4,
             resync=0),
        # a region of interest of no round size, a z-block per slice, an odd number of
        # bins and views
        dict(name="ragged", kind="icd", N=222, Nz=10, views=363, threads=64, omp=5, iters=3,
             resync=0),
        # the 4D interlaced scan (256^2 x 16 in 16 frames, 2048 views)
        dict(name="frames", kind="icd", N=256, Nz=16, views=2048, frames=16, threads=64,
             lines=512, omp=32, iters=4, resync=1),
        # edge-only updates of a reconstruction that has settled elsewhere
        dict(name="edges", kind="icd", N=384, Nz=16, views=512, threads=256, omp=8, iters=2,
             resync=1, edge=True),
        # phase-contrast tomography, few lines in flight (its footprints couple more)
        dict(name="phase", kind="icd", N=192, Nz=16, views=240, threads=256, lines=144, omp=8,
             iters=2, resync=0, pc=True),
        # a coarse multi-resolution stage of the production slab: voxels of six bins
        dict(name="coarse", kind="icd", N=128, Nz=32, factor=4, views=1024, threads=256,
             lines=256, omp=32, iters=2, resync=0, I0=1e4),
        # several small slabs of a batch, thin ones among them
        dict(name="batch", kind="batch", slabs="128x4x180,192x16x360,256x8x360,384x4x720",
             threads=64, omp=16, iters=2, resync=1),
        # the filtered-backprojection start of the production slab
        dict(name="fbp", kind="fbp", N=512, Nz=32, views=1024, threads=256, omp=32),
        # the warm-start network on the production slab, and one gradient at the shape
        # that it is trained on
        dict(name="infer", kind="infer", d0=512, d1=512, d2=32),
        dict(name="train", kind="train", d0=256, d1=256, d2=16),
        # one ring-offset update of a small detector: the smallest call
        dict(name="offset", kind="offset", views=256, bins=192, rows=8),
    ]


def _log_int(rng, lo, hi, step=1):
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(lo, int(round(n / step)) * step))


def draw(rng):
    kind = rng.choice(["icd", "icd", "icd", "frames", "edge", "pc", "coarse", "batch", "fbp",
                       "infer", "train", "offset"])
    if kind in ("icd", "edge", "pc"):
        pc = kind == "pc"
        c = dict(kind="icd", N=_log_int(rng, 64, 256 if pc else 512, 2),
                 Nz=rng.randint(4, 16 if pc else 32), views=_log_int(rng, 90, 400 if pc else 1024),
                 threads=256 if pc else rng.choice([64, 256]), omp=rng.choice([2, 4, 8, 16, 32]),
                 iters=2, resync=rng.choice([0, 1]))
        if kind != "icd":
            c[kind] = True
        if pc:
            c["lines"] = max(16, c["N"] ** 2 // 256)
        return c
    if kind == "frames":
        f = rng.choice([2, 3, 4, 6, 8, 12, 16])
        return dict(kind="icd", N=_log_int(rng, 96, 256, 2), Nz=rng.randint(4, 16), frames=f,
                    views=f * rng.randint(64, 128), threads=rng.choice([64, 256]),
                    omp=rng.choice([4, 16, 32]), iters=4, resync=1)
    if kind == "coarse":
        n = _log_int(rng, 64, 160, 2)
        return dict(kind="icd", N=n, Nz=rng.randint(4, 32), factor=rng.choice([2, 4]),
                    views=_log_int(rng, 180, 1000), threads=256, lines=max(16, n * n // 128),
                    omp=rng.choice([8, 32]), iters=2, resync=0, I0=1e4)
    if kind == "batch":
        slabs = ",".join("%dx%dx%d" % (rng.choice([128, 192, 256, 384]), rng.choice([4, 8, 16]),
                                       rng.choice([180, 360, 720])) for _ in range(rng.randint(2, 5)))
        return dict(kind="batch", slabs=slabs, threads=64, omp=16, iters=2, resync=1)
    if kind == "fbp":
        return dict(kind="fbp", N=_log_int(rng, 96, 512, 2), Nz=rng.randint(4, 32),
                    views=_log_int(rng, 180, 1024), threads=256, omp=rng.choice([4, 32]))
    if kind == "infer":
        return dict(kind="infer", d0=_log_int(rng, 64, 512, 8), d1=_log_int(rng, 64, 512, 8),
                    d2=_log_int(rng, 8, 32, 8))
    if kind == "train":
        return dict(kind="train", d0=_log_int(rng, 64, 256, 8), d1=_log_int(rng, 64, 256, 8),
                    d2=_log_int(rng, 8, 32, 8))
    return dict(kind="offset", views=_log_int(rng, 180, 1024), bins=_log_int(rng, 96, 768),
                rows=_log_int(rng, 4, 64))


# -- scans ------------------------------------------------------------------
def _config(case, N=None, Nz=None, views=None):
    T = case.get("frames", 1)
    return dataclasses.replace(
        synth.C1, name="case", N_xy=N or case["N"], N_z=Nz or case["Nz"],
        N_p=views or case["views"], mult_xy=1.5 * case.get("factor", 1), N_time=T, I0=case.get("I0", 2e4),
        num_threads=case["omp"], interlaced_K=8 if T > 1 else 0,
        interlaced_N_theta=512 if T > 1 else 0, motion_per_frame=case.get("motion", 0.5) if T > 1 else 0.0)


def _frame_of_view(cfg, times):
    r0, rd = cfg.rtime()
    return np.clip(np.floor((times - r0) / rd), 0, cfg.N_time - 1).astype(np.int64)


def _ellipsoids(cfg, rng):
    """(centre x, y, z, semi-axes a, b, c, angle, attenuation, direction), lengths in
    detector pixels (z in slices), x and y from the rotation axis."""
    L, nz, out = cfg.N_xy * cfg.mult_xy, cfg.N_z, []
    for _ in range(10):
        r, t = 0.32 * L * math.sqrt(rng.uniform()), rng.uniform(0, 2 * math.pi)
        out.append((r * math.cos(t), r * math.sin(t), rng.uniform(0.2, 0.8) * nz,
                    rng.uniform(0.05, 0.2) * L, rng.uniform(0.05, 0.2) * L,
                    rng.uniform(0.3, 0.8) * nz, rng.uniform(0, math.pi),
                    rng.uniform(cfg.mu_lo, cfg.mu_hi), rng.uniform(0, 2 * math.pi)))
    return out


def _scale2(cfg, e):
    """1 - ((z - cz) / c)^2 of every slice, at least 0."""
    z = torch.arange(cfg.N_z, device="cuda") + 0.5
    return (1 - ((z - e[2]) / e[5]) ** 2).clamp_(min=0)


def _phantom(cfg, ells):
    """[N_time][N_z][N_y][N_x] float32."""
    x = (torch.arange(cfg.N_xy, device="cuda") + 0.5 - cfg.N_xy / 2) * cfg.mult_xy
    vol = torch.zeros((cfg.N_time, cfg.N_z, cfg.N_xy, cfg.N_xy), device="cuda")
    for f in range(cfg.N_time):
        m = cfg.motion_per_frame * cfg.mult_xy * f
        for e in ells:
            dx, dy = x[None, :] - e[0] - m * math.cos(e[8]), x[:, None] - e[1] - m * math.sin(e[8])
            u = (dx * math.cos(e[6]) + dy * math.sin(e[6])) / e[3]
            v = (dy * math.cos(e[6]) - dx * math.sin(e[6])) / e[4]
            vol[f] += e[7] * ((u * u + v * v)[None] < _scale2(cfg, e)[:, None, None])
    return vol


def _line_integrals(cfg, ells):
    """[N_p][N_r][N_t] float32: the ellipsoids' projections r = x cos - y sin."""
    ang, times = cfg.views()
    th = torch.tensor(np.deg2rad(ang), device="cuda")
    frame = torch.tensor(_frame_of_view(cfg, times), device="cuda")
    r = torch.arange(cfg.N_r, device="cuda") + 0.5 - cfg.N_r / 2
    ax = torch.zeros((cfg.N_p, cfg.N_r, cfg.N_z), device="cuda")
    for e in ells:
        m = cfg.motion_per_frame * cfg.mult_xy * frame
        cx, cy = e[0] + m * math.cos(e[8]), e[1] + m * math.sin(e[8])
        s = (cx * th.cos() - cy * th.sin()).float()
        al = th + e[6]  # angle of the ray normal (cos, -sin) from the first semi-axis
        w2 = ((e[3] * al.cos()) ** 2 + (e[4] * al.sin()) ** 2).float()[:, None, None]
        t2 = (r[None, :] - s[:, None])[:, :, None] ** 2
        ax += (2 * e[7] * e[3] * e[4]) * (w2 * _scale2(cfg, e) - t2).clamp_(min=0).sqrt() / w2
    return ax


class _Scan:
    """y, w (counts) and the true ring offsets of one seeded scan, and a volume and
    offsets to restart from: the phantom, a little blurred, with noise."""

    def __init__(self, cfg, seed, pc=False):
        rng = np.random.default_rng(seed)
        gen = torch.Generator("cuda").manual_seed(seed)
        ells = _ellipsoids(cfg, rng)
        self.cfg, self.phantom = cfg, _phantom(cfg, ells)
        ax = _line_integrals(cfg, ells)
        if pc:  # the engine's detector Laplacian (pitch 1) of the projections
            k = torch.tensor([[-.5, -1, -.5], [-1, 6, -1], [-.5, -1, -.5]], device="cuda")
            p = torch.nn.functional.pad(ax, (1, 1, 1, 1))
            ax = sum(k[i, j] * p[:, i:i + cfg.N_r, j:j + cfg.N_t] for i in range(3) for j in range(3))
        self.d = cfg.offset_sigma * torch.randn((cfg.N_r, cfg.N_t), generator=gen, device="cuda")
        self.w = torch.poisson(cfg.I0 * torch.exp(-(ax + self.d)), generator=gen).clamp_(min=1)
        self.y = torch.log(cfg.I0 / self.w)
        zing = torch.rand(self.y.shape, generator=gen, device="cuda") < cfg.zinger_frac
        self.y[zing] = cfg.zinger_scale * self.y.max()
        half = torch.nn.functional.avg_pool2d(self.phantom, 2)
        up = torch.nn.functional.interpolate(half, size=(cfg.N_xy, cfg.N_xy), mode="bilinear")
        up = 0.75 * self.phantom + 0.25 * up
        sd = 0.01 * float(self.phantom.max())
        self.start = (up + sd * torch.randn(up.shape, generator=gen, device="cuda")).clamp_(min=0)
        self.d0 = self.d + 0.1 * cfg.offset_sigma * torch.randn(self.d.shape, generator=gen,
                                                                device="cuda")


class _Recon:
    """An Engine over a scan and its open Icd state, closed when dropped."""

    def __init__(self, case, scan):
        cfg = scan.cfg
        args = cfg.cli_args()
        if case.get("edge"):
            args.append("--only_Edge_Updates")
        run = tempfile.mkdtemp(prefix="xt_case_")
        try:
            ang, t = cfg.views()
            synth.write_view_info(run, ang, t)
            self.eng = xt_hip.Engine(run, args, read_sinogram=False)
        finally:
            shutil.rmtree(run, ignore_errors=True)
        self.icd = None
        torch.from_numpy(self.eng.sino("Projection")).copy_(scan.y)
        torch.from_numpy(self.eng.sino("Weight")).copy_(scan.w)
        self.start, self.d0 = scan.start.cpu().numpy(), scan.d0.cpu().numpy()
        if case["kind"] in ("icd", "batch"):
            self.put_start()
        xt_hip.set_option(xt_hip.OPT_AUTOTUNE, 0)
        xt_hip.set_option(xt_hip.OPT_LINES, case.get("lines", 0))
        xt_hip.set_option(xt_hip.OPT_LINE_THREADS, case["threads"])
        xt_hip.set_option(xt_hip.OPT_PHASE_CONTRAST, 1 if case.get("pc") else 0)
        xt_hip.set_option(xt_hip.OPT_RESYNC_EVERY, case.get("resync", 0))
        self.icd = xt_hip.Icd(self.eng)

    def put_start(self):
        self.eng.set_volume(self.start)
        self.eng.offset()[:] = self.d0

    def result(self):
        return {"object": self.eng.volume(), "offset": self.eng.offset().copy()}

    def __del__(self):
        if getattr(self, "icd", None) is not None:
            self.icd.close()
        if getattr(self, "eng", None) is not None:
            self.eng.close()


class _Batch:
    def __init__(self, case, seed):
        self.recons = []
        for k, s in enumerate(case["slabs"].split(",")):
            n, nz, views = (int(v) for v in s.split("x"))
            self.recons.append(_Recon(case, _Scan(_config(case, n, nz, views), seed * 16 + k)))
        self.batch = xt_hip.IcdBatch([r.icd for r in self.recons])

    def __del__(self):
        if getattr(self, "batch", None) is not None:
            self.batch.close()


class _Net:
    """The committed network at a shape, with a noisy volume and its target on the GPU."""

    def __init__(self, case, seed):
        d = (case["d0"], case["d1"], case["d2"])
        self.net = xt_hip.UNet.load(WEIGHTS, d, train=case["kind"] == "train")
        self.x, self.target = _volumes(case, seed)
        self.out = torch.empty_like(self.x)
        self.grad = np.zeros(self.net.n, np.float32)

    def __del__(self):
        if getattr(self, "net", None) is not None:
            self.net.close()


def _volumes(case, seed):
    """(a streaky volume such as a filtered backprojection gives, the volume behind it),
    float32 [d0][d1][d2] on the GPU, attenuation around 1e-3."""
    d = (case["d0"], case["d1"], case["d2"])
    rng, gen = np.random.default_rng(seed), torch.Generator("cuda").manual_seed(seed)
    g = [torch.arange(n, device="cuda") + 0.5 for n in d]
    vol = torch.zeros(d, device="cuda")
    for _ in range(8):
        c = [rng.uniform(0.25, 0.75) * n for n in d]
        a = [rng.uniform(0.08, 0.3) * n for n in d]
        q = [((g[i] - c[i]) / a[i]) ** 2 for i in range(3)]
        vol[(q[0][:, None, None] + q[1][None, :, None] + q[2][None, None, :]) < 1] = \
            rng.uniform(0.5e-3, 2e-3)
    return vol + 3e-4 * torch.randn(d, generator=gen, device="cuda"), vol


def _offset_arrays(case, seed):
    """Error sinogram (noise, ring offsets, some zingers), weights and offsets."""
    n = (case["views"], case["bins"], case["rows"])
    gen = torch.Generator("cuda").manual_seed(seed)
    w = torch.poisson(torch.full(n, 5e3, device="cuda"), generator=gen).clamp_(min=1)
    e = torch.randn(n, generator=gen, device="cuda") / w.sqrt()
    e += 0.01 * torch.randn(n[1:], generator=gen, device="cuda")
    e[torch.rand(n, generator=gen, device="cuda") < 0.005] += 1.0
    return e, w, torch.zeros(n[1:], device="cuda")


# -- what is timed ----------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        s = _Batch(case, seed)
    elif kind in ("infer", "train"):
        s = _Net(case, seed)
    elif kind == "offset":
        s = _offset_arrays(case, seed)
    else:
        s = _Recon(case, _Scan(_config(case), seed, bool(case.get("pc"))))
    torch.cuda.synchronize()
    return case, s


def run(state):
    case, s = state
    kind = case["kind"]
    if kind == "icd":
        s.put_start()
        s.icd.upload()
        s.icd.iterate(case["iters"])
        s.icd.download()
        return s.result()
    if kind == "fbp":
        s.icd.fbp()
        s.icd.download()
        return s.result()
    if kind == "batch":
        for r in s.recons:
            r.put_start()
            r.icd.upload()
        s.batch.iterate(case["iters"])
        for r in s.recons:
            r.icd.download()
        return [r.result() for r in s.recons]
    L = xt_hip.lib()
    if kind == "infer":
        xt_hip._check(L.xt_unet_forward(s.net.h, s.x.data_ptr(), s.out.data_ptr()))
        return s.out
    if kind == "train":
        loss = ctypes.c_double()
        xt_hip._check(L.xt_unet_loss_grad(s.net.h, s.x.data_ptr(), s.target.data_ptr(),
                                          ctypes.byref(loss), s.grad.ctypes.data))
        return {"loss": np.float64(loss.value), "grad": s.grad}
    e, w, d = s
    xt_hip.offset_update_noalloc(*e.shape, 4.0, 0.1, True, e.data_ptr(), w.data_ptr(), d.data_ptr())
    return {"e": e, "offset": d}


def _scan_work(cfg, iters):
    """One pass over the sinogram (y and w) and the object (in and out); per voxel and
    view that an iteration updates, the two sums over a column of (mult_xy + 1) bins and
    its correction of e, ten operations an entry."""
    sino, obj = cfg.N_p * cfg.N_r * cfg.N_t, cfg.N_time * cfg.N_z * cfg.N_xy ** 2
    entries = obj * (cfg.N_p / cfg.N_time) * (cfg.mult_xy + 1) * cfg.mult_z
    return {"bytes": 8.0 * sino + 8.0 * obj + 8.0 * cfg.N_r * cfg.N_t,
            "flops": 10.0 * entries * iters}


def work(case):
    kind = case["kind"]
    if kind == "offset":
        n = case["views"] * case["bins"] * case["rows"]
        return {"bytes": 12.0 * n + 8.0 * case["bins"] * case["rows"], "flops": 8.0 * n}
    if kind in ("infer", "train"):
        v = case["d0"] * case["d1"] * case["d2"]
        f = sum(54.0 * ci * co * v / 8 ** lvl for lvl, ci, co in CONVS)
        n = sum(co * (27 * ci + 1) for _, ci, co in CONVS) + 17
        return {"bytes": 8.0 * v + 4.0 * n * (2 if kind == "train" else 1),
                "flops": f * (3 if kind == "train" else 1)}
    if kind == "batch":
        ws = [_scan_work(_config(case, *(int(v) for v in s.split("x"))), case["iters"])
              for s in case["slabs"].split(",")]
        return {k: sum(w[k] for w in ws) for k in ws[0]}
    cfg = _config(case)
    if kind == "fbp":  # the filter by transforms, two samples of the rows per voxel and view
        w = _scan_work(cfg, 0)
        w["bytes"] -= 4.0 * (cfg.N_p * cfg.N_r * cfg.N_t + cfg.N_z * cfg.N_xy ** 2)
        w["flops"] = 4.0 * cfg.N_z * cfg.N_xy ** 2 * cfg.N_p
        return w
    w = _scan_work(cfg, case["iters"])
    if case.get("pc"):  # the Laplacian of a column: two more bins, three rows
        w["flops"] *= 3.0 * (cfg.mult_xy + 3) / (cfg.mult_xy + 1)
    return w


# -- 64-bit values ----------------------------------------------------------
def exact(case, seed):
    """run()'s outputs in 64 bits where they are functions of the inputs alone; an ICD
    iteration's depend on which lines are in flight together."""
    kind = case["kind"]
    if kind == "offset":
        return _exact_offset(case, seed)
    if kind == "fbp":
        return _exact_fbp(case, seed)
    if kind == "infer":
        x, _ = _volumes(case, seed)
        with torch.no_grad():
            return _network(x.double(), _parameters())
    if kind == "train":
        x, t = _volumes(case, seed)
        p = _parameters().requires_grad_()
        scale = _scale()
        loss = ((_network(x.double(), p) - t.double()) * scale).square().mean()
        loss.backward()
        return {"loss": float(loss), "grad": p.grad.cpu().numpy()}
    return None


def _exact_offset(case, seed):
    e, w, d = (a.double() for a in _offset_arrays(case, seed))
    small = e * e * w < 16.0
    t = 0.4 * w.sqrt()
    num = torch.where(small, e * w, t * e.sign()).sum(0)
    den = torch.where(small, w, t / e.abs()).sum(0)
    gamma = (d + num / den).sum() / (1 / den).sum()
    step = (num - gamma) / den
    return {"e": e - step, "offset": d + step}


def _exact_fbp(case, seed):
    scan = _Scan(_config(case), seed)
    cfg, y = scan.cfg, scan.y.double()
    sd = (y.square().mean(0) - y.mean(0).square()).clamp(min=0).sqrt()
    keep = (y - y.mean(0)).abs() <= 4 * sd
    m = (y * keep).sum(0) / keep.sum(0)
    i = torch.arange(cfg.N_r, device="cuda")
    trend = sum(m[(i + k).clamp(0, cfg.N_r - 1)] for k in range(-7, 8)) / 15
    d = m - trend
    d = d - d.mean()
    p = y - d
    mid = torch.stack((p[:, :-2], p[:, 1:-1], p[:, 2:])).median(0).values
    p = torch.cat((p[:, :1], mid, p[:, -1:]), 1)
    # Ram-Lak taps: 1/4 at 0, -1/(n pi)^2 at odd n
    n = torch.arange(-(cfg.N_r - 1), cfg.N_r, device="cuda", dtype=torch.float64)
    taps = torch.where(n % 2 != 0, -1 / (n * math.pi) ** 2, torch.zeros_like(n))
    taps[cfg.N_r - 1] = 0.25
    size = 4 * cfg.N_r
    q = torch.fft.irfft(torch.fft.rfft(p, size, 1) * torch.fft.rfft(taps, size)[None, :, None],
                        size, 1)[:, cfg.N_r - 1:2 * cfg.N_r - 1]
    ang = np.deg2rad(cfg.views()[0])
    order = np.argsort(ang % math.pi)
    s = (ang % math.pi)[order]
    wv = np.empty(cfg.N_p)
    wv[order] = 0.5 * (np.append(s[1:], s[0] + math.pi) - np.append(s[-1] - math.pi, s[:-1]))
    g = (torch.arange(cfg.N_xy, device="cuda", dtype=torch.float64) + 0.5 - cfg.N_xy / 2) * cfg.mult_xy
    vol = torch.zeros((cfg.N_xy ** 2, cfg.N_t), device="cuda", dtype=torch.float64)
    pad = torch.nn.functional.pad(q, (0, 0, 1, 1))  # zero beyond the detector
    for v in range(cfg.N_p):
        u = (g[None, :] * math.cos(ang[v]) - g[:, None] * math.sin(ang[v])).reshape(-1)
        u = u + cfg.N_r / 2 - 0.5
        f = u.floor()
        k = f.long() + 1
        ok = ((k >= 0) & (k <= cfg.N_r))[:, None]
        k = k.clamp(0, cfg.N_r)
        fr = (u - f)[:, None]
        vol += wv[v] * torch.where(ok, (1 - fr) * pad[v][k] + fr * pad[v][k + 1], 0.0)
    vol = vol.reshape(cfg.N_xy, cfg.N_xy, cfg.N_t).permute(2, 0, 1)
    return {"object": vol[None].contiguous(), "offset": d}


def _scale():
    with np.load(WEIGHTS, allow_pickle=False) as z:
        return float(z["scale"])


def _parameters():
    with np.load(WEIGHTS, allow_pickle=False) as z:
        return torch.tensor(z["params"].astype(np.float64), device="cuda")


def _network(x, params):
    """The network (include/xt_unet.h) on a float64 volume [d0][d1][d2]."""
    pos, scale = 0, _scale()

    def take(*shape):
        nonlocal pos
        n = math.prod(shape)
        pos += n
        return params[pos - n:pos].reshape(shape)

    def conv(t, k):
        _, ci, co = CONVS[k]
        w, b = take(co, 27, ci), take(co)
        d = t.shape[:3]
        p = torch.nn.functional.pad(t, (0, 0, 1, 1, 1, 1, 1, 1))
        out = b.expand(math.prod(d), co)
        for tap in range(27):
            a, e, f = tap // 9, tap // 3 % 3, tap % 3
            part = p[a:a + d[0], e:e + d[1], f:f + d[2]].reshape(-1, ci)
            out = out + part @ w[:, tap].t()
        return out.reshape(*d, co).relu()

    def pool(t):
        d = t.shape
        return t.reshape(d[0] // 2, 2, d[1] // 2, 2, d[2] // 2, 2, d[3]).mean((1, 3, 5))

    def up(low, skip):
        for i in range(3):
            low = low.repeat_interleave(2, i)
        return torch.cat((low, skip), 3)

    e1 = conv(conv((x * scale)[..., None], 0), 1)
    e2 = conv(conv(pool(e1), 2), 3)
    e3 = conv(conv(pool(e2), 4), 5)
    t = conv(conv(pool(e3), 6), 7)
    t = conv(conv(up(t, e3), 8), 9)
    t = conv(conv(up(t, e2), 10), 11)
    t = conv(conv(up(t, e1), 12), 13)
    h = (t @ take(16)) + take(1)
    return (x * scale + h) / scale
