// xt_unet.hip -- the learned warm start: a 3D U-Net (4 levels, channels
// 16/32/64/128, 3x3x3 convs) trained and run by this library's own kernels.
//
// Activations are channels-last bf16 [V][C] over V = d0*d1*d2 voxels (d2
// fastest), so the 8 consecutive channels one MFMA lane feeds are one 16-byte
// load.  Every 3x3x3 conv is an implicit GEMM on v_mfma_f32_16x16x32_bf16 with
// FP32 accumulation:
//   forward        out[v][co] = sum_{tap,ci} in[v+off(tap)][ci] * W[co][tap][ci]
//   backward-data  gin[v][ci] = sum_{tap,co} gout[v+off(tap)][co] * W[co][26-tap][ci]
//                  (the same kernel with the flipped, transposed weights)
//   weight grad    dW[co][tap*Ci+ci] = sum_v gout[v][co] * in[v+off(tap)][ci]
//                  (split over voxel chunks, FP32 atomics)
// FP32 master weights with Adam; bf16 copies of both weight layouts are
// regenerated after every update.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <random>
#include <vector>

#include "xt_unet_internal.h"

typedef uint16_t bf16_t;  // raw bfloat16 bits
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

#define UN_HIP(call)                                                                         \
  do {                                                                                       \
    hipError_t _e = (call);                                                                  \
    if (_e != hipSuccess)                                                                    \
      return xt_report_error(XT_E_HIP, "%s failed: %s (%s:%d)", #call, hipGetErrorString(_e), \
                             __FILE__, __LINE__);                                            \
  } while (0)
#define UN_TRY(expr)               \
  do {                             \
    int _rc = (expr);              \
    if (_rc != XT_OK) return _rc;  \
  } while (0)

// float -> bf16, round to nearest even (finite inputs)
__device__ __host__ inline bf16_t f2bf(float f) {
  uint32_t u;
  memcpy(&u, &f, 4);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (bf16_t)(u >> 16);
}
__device__ inline float bf2f(bf16_t b) { return __uint_as_float((uint32_t)b << 16); }
// ReLU mask of a stored activation: strictly positive
__device__ inline bool bf_pos(bf16_t b) { return b != 0 && !(b & 0x8000u); }

__device__ inline bf16x8 as_bf16x8(uint4 q) { return __builtin_bit_cast(bf16x8, q); }

// ---------------------------------------------------------------------------
// 3x3x3 conv, forward (also backward-data).  Workgroup = 4 waves; a wave
// computes 16*MB voxels x 16*NB output channels.  K runs over kk = tap*Ci + ci
// padded to Kpad (multiple of 32) with zero weights; Ci % 8 == 0 (one 16-byte load
// per lane and fragment).  Optional epilogue: + bias, ReLU, x (mask > 0).
template <int MB, int NB>
__global__ void __launch_bounds__(256) k_conv3(const bf16_t *__restrict__ in, int Ci,
                                               const bf16_t *__restrict__ W, int Kpad,
                                               const float *__restrict__ bias, int Co, int d0,
                                               int d1, int d2, bf16_t *__restrict__ out, int relu,
                                               const bf16_t *__restrict__ mask) {
  const int V = d0 * d1 * d2, P = d1 * d2;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int m0 = (blockIdx.x * 4 + wave) * (16 * MB);
  const int n0 = blockIdx.y * (16 * NB);
  if (m0 >= V) return;
  int c0[MB], c1[MB], c2[MB];
#pragma unroll
  for (int mb = 0; mb < MB; mb++) {
    const int v = m0 + mb * 16 + r;
    c0[mb] = v < V ? v / P : -100;  // out-of-range rows never pass the bounds test
    c1[mb] = (v / d2) % d1;
    c2[mb] = v % d2;
  }
  f32x4 acc[MB][NB];
#pragma unroll
  for (int mb = 0; mb < MB; mb++)
#pragma unroll
    for (int nb = 0; nb < NB; nb++) acc[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint4 zero4 = {0u, 0u, 0u, 0u};
  int tap = (g * 8) / Ci, ci = g * 8 - tap * Ci;  // (tap, ci) of kk = k0 + g*8
  for (int k0 = 0; k0 < Kpad; k0 += 32) {
    bf16x8 a[MB], b[NB];
    const int a0 = tap / 9 - 1, a1 = (tap / 3) % 3 - 1, a2 = tap % 3 - 1;
    const bool tok = tap < 27;
    const int off = a0 * P + a1 * d2 + a2;
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
      const int p0 = c0[mb] + a0, p1 = c1[mb] + a1, p2 = c2[mb] + a2;
      const bool ok = tok && (unsigned)p0 < (unsigned)d0 && (unsigned)p1 < (unsigned)d1 &&
                      (unsigned)p2 < (unsigned)d2;
      const int v = m0 + mb * 16 + r;
      a[mb] = as_bf16x8(ok ? *(const uint4 *)(in + (size_t)(v + off) * Ci + ci) : zero4);
    }
    ci += 32;
    while (ci >= Ci) {
      ci -= Ci;
      tap++;
    }
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
      const int co = n0 + nb * 16 + r;
      b[nb] = as_bf16x8(co < Co ? *(const uint4 *)(W + (size_t)co * Kpad + k0 + g * 8) : zero4);
    }
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
      for (int nb = 0; nb < NB; nb++)
        acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[mb], b[nb], acc[mb][nb], 0, 0, 0);
  }
  // accumulator lane layout: column (output channel) r, rows (voxels) g*4 + i
#pragma unroll
  for (int nb = 0; nb < NB; nb++) {
    const int co = n0 + nb * 16 + r;
    if (co >= Co) continue;
    const float bv = bias ? bias[co] : 0.f;
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int v = m0 + mb * 16 + g * 4 + i;
        if (v >= V) continue;
        float val = acc[mb][nb][i] + bv;
        if (relu) val = fmaxf(val, 0.f);
        if (mask && !bf_pos(mask[(size_t)v * Co + co])) val = 0.f;
        out[(size_t)v * Co + co] = f2bf(val);
      }
  }
}

// LDS-tiled variant for Ci % 32 == 0: a workgroup's 64*MB voxels form a TY x TX
// tile of one d0-plane (TX along d2); per chunk of 32 input channels the tile
// and its one-voxel halo in d0, d1 and d2 are staged in LDS once and every
// tap's A fragment is read from there (the direct kernel reads each input 27
// times from L2).  K order: channel chunks outer, taps inner, one tap per MFMA
// K-step.  TY | d1 and TX | d2.
template <int MB, int NB>
__global__ void __launch_bounds__(256) k_conv3_lds(const bf16_t *__restrict__ in, int Ci,
                                                   const bf16_t *__restrict__ W, int Kpad,
                                                   const float *__restrict__ bias, int Co, int d0,
                                                   int d1, int d2, int TY, int TX,
                                                   bf16_t *__restrict__ out, int relu,
                                                   const bf16_t *__restrict__ mask) {
  constexpr int CC = 32, CP = CC + 8;  // channels of a chunk, padded stride of a staged voxel
  extern __shared__ uint4 lds4[];
  bf16_t *tile = (bf16_t *)lds4;  // [3][TY+2][TX+2][CP]
  const int P = d1 * d2;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.y * (16 * NB);
  const int ntx = d2 / TX, nty = d1 / TY;
  int bi = blockIdx.x;
  const int bx = bi % ntx;
  bi /= ntx;
  const int by = bi % nty;
  const int p0 = bi / nty;
  const int y0 = by * TY, x0 = bx * TX;
  const int HY = TY + 2, HX = TX + 2, HV = 3 * HY * HX;
  int ty[MB], tx[MB];
  bool rok[MB];
#pragma unroll
  for (int mb = 0; mb < MB; mb++) {
    const int m = (wave * MB + mb) * 16 + r;
    ty[mb] = m / TX;
    tx[mb] = m % TX;
    rok[mb] = ty[mb] < TY;
  }
  f32x4 acc[MB][NB];
#pragma unroll
  for (int mb = 0; mb < MB; mb++)
#pragma unroll
    for (int nb = 0; nb < NB; nb++) acc[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint4 zero4 = {0u, 0u, 0u, 0u};
  for (int c0 = 0; c0 < Ci; c0 += CC) {
    __syncthreads();  // the previous chunk's fragments are read
    for (int q = threadIdx.x; q < HV * (CC / 8); q += 256) {
      const int hv = q / (CC / 8), c8 = q % (CC / 8);
      const int hz = hv / (HY * HX), rem = hv % (HY * HX);
      const int pp = p0 + hz - 1, yy = y0 + rem / HX - 1, xx = x0 + rem % HX - 1;
      uint4 v = zero4;
      if ((unsigned)pp < (unsigned)d0 && (unsigned)yy < (unsigned)d1 && (unsigned)xx < (unsigned)d2)
        v = *(const uint4 *)(in + ((size_t)pp * P + (size_t)yy * d2 + xx) * Ci + c0 + 8 * c8);
      *(uint4 *)(tile + (size_t)hv * CP + 8 * c8) = v;
    }
    __syncthreads();
    for (int tap = 0; tap < 27; tap++) {
      const int cg = g * 8;
      const int a0 = tap / 9, a1 = (tap / 3) % 3, a2 = tap % 3;  // halo offsets 0..2
      bf16x8 a[MB], b[NB];
#pragma unroll
      for (int mb = 0; mb < MB; mb++) {
        const int hv = (a0 * HY + ty[mb] + a1) * HX + tx[mb] + a2;
        a[mb] = as_bf16x8(rok[mb] ? *(const uint4 *)(tile + (size_t)hv * CP + cg) : zero4);
      }
#pragma unroll
      for (int nb = 0; nb < NB; nb++) {
        const int co = n0 + nb * 16 + r;
        b[nb] = as_bf16x8(co < Co
                              ? *(const uint4 *)(W + (size_t)co * Kpad + (size_t)tap * Ci + c0 + cg)
                              : zero4);
      }
#pragma unroll
      for (int mb = 0; mb < MB; mb++)
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
          acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[mb], b[nb], acc[mb][nb], 0, 0, 0);
    }
  }
#pragma unroll
  for (int nb = 0; nb < NB; nb++) {
    const int co = n0 + nb * 16 + r;
    if (co >= Co) continue;
    const float bv = bias ? bias[co] : 0.f;
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int m = (wave * MB + mb) * 16 + g * 4 + i;
        const int yy = m / TX, xx = m % TX;
        if (yy >= TY) continue;
        const size_t v = ((size_t)p0 * d1 + y0 + yy) * d2 + x0 + xx;
        float val = acc[mb][nb][i] + bv;
        if (relu) val = fmaxf(val, 0.f);
        if (mask && !bf_pos(mask[v * Co + co])) val = 0.f;
        out[v * Co + co] = f2bf(val);
      }
  }
}

// 3x3x3 conv of Ci = 16 * NC channels (NC 1 or 3: the layers at full resolution, forward
// and backward-data): a workgroup keeps 16 * NC x 16 weights in registers and marches along
// d0 over a tile of TY x TX voxels (256 of them, TX = 1 << ltx along d2).  The input planes
// p-1, p, p+1 with their halo lie in a ring of four in LDS, so each is read once per tile
// (4/3 of the voxels, not 27 times or 3 * 4/3) while the one after next is under way to
// registers; halves of 8 channels are laid out apart, so that a fragment's 16 voxels are
// 256 consecutive bytes.  K order: chunks of 16 channels, in each the taps by pairs, as
// k_conv3 with Ci = 16 (bit for bit the same sums).  The product is taken as weights x
// voxels: a lane ends with 4 channels of one voxel and stores them together.  Bound by
// the LDS reads of fragments (one per MFMA, 8 cycles of a CU each).  512 x 512 x 32:
//   48->16   755 us; 1580 with a tile of one plane staged per channel chunk (3 * 4/3 reads)
//   16->16   180 us; 521 with fragments read from L2 for every tap
constexpr int MARCH_HV = 344;  // staged voxels of a plane, at most 340, up to a half's stride

template <int NC>
__global__ void __launch_bounds__(512, 2) k_conv3_march(
    const bf16_t *__restrict__ in, const bf16_t *__restrict__ W, int Kpad,
    const float *__restrict__ bias, int Co, int d0, int d1, int d2, int ltx, int seg,
    bf16_t *__restrict__ out, int relu, const bf16_t *__restrict__ mask) {
  constexpr int Ci = 16 * NC, C8 = 2 * NC, PL = C8 * MARCH_HV, NP = (340 * C8 + 511) / 512;
  extern __shared__ uint4 ring[];  // [4][C8][MARCH_HV]
  const int TX = 1 << ltx, TY = 256 >> ltx, HX = TX + 2, HV = (TY + 2) * HX, P = d1 * d2;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, g = lane >> 4;
  const bool odd = g >> 1;  // the second tap of a pair
  const int ntx = d2 >> ltx;
  const int x0 = (blockIdx.x % ntx) << ltx, y0 = blockIdx.x / ntx * TY;
  const int n0 = blockIdx.y * 16;
  const int pb = blockIdx.z * seg, pe = min(pb + seg, d0);
  const uint4 zero4 = {0u, 0u, 0u, 0u};
  // this thread's pieces (8 channels of a voxel) of a plane
  int pix[NP], dst[NP];
#pragma unroll
  for (int i = 0; i < NP; i++) {
    const int q = tid + i * 512, hv = q / C8, c8 = q - hv * C8;
    const int yy = y0 + hv / HX - 1, xx = x0 + hv % HX - 1;
    const bool ok = hv < HV && (unsigned)yy < (unsigned)d1 && (unsigned)xx < (unsigned)d2;
    pix[i] = ok ? yy * d2 + xx : -1;
    dst[i] = hv < HV ? c8 * MARCH_HV + hv : -1;
  }
  uint4 v[NP];
  auto load = [&](int p) {
#pragma unroll
    for (int i = 0; i < NP; i++) {
      v[i] = zero4;
      if ((unsigned)p < (unsigned)d0 && pix[i] >= 0)
        v[i] = *(const uint4 *)(in + (size_t)(p * P + pix[i]) * Ci + (tid + i * 512) % C8 * 8);
    }
  };
  auto store = [&](int p) {
#pragma unroll
    for (int i = 0; i < NP; i++)
      if (dst[i] >= 0) ring[((p + 4) & 3) * PL + dst[i]] = v[i];
  };
  for (int p = pb - 1; p <= pb + 1; p++) {
    load(p);
    store(p);
  }
  uint4 w[NC][14];
#pragma unroll
  for (int c = 0; c < NC; c++)
#pragma unroll
    for (int s = 0; s < 14; s++) {
      const int tap = 2 * s + odd;
      w[c][s] = tap < 27 ? *(const uint4 *)(W + (size_t)(n0 + r) * Kpad + tap * Ci + c * 16 + (g & 1) * 8)
                         : zero4;
    }
  // the wave's two blocks of 16 voxels, hv of their taps' first corner
  const int m0 = wave * 32 + r, m1 = m0 + 16;
  const int hv0 = (m0 >> ltx) * HX + (m0 & (TX - 1)), hv1 = (m1 >> ltx) * HX + (m1 & (TX - 1));
  const int base = (g & 1) * MARCH_HV + hv0, step = hv1 - hv0;
  float bv[4] = {0.f, 0.f, 0.f, 0.f};
  if (bias)
#pragma unroll
    for (int i = 0; i < 4; i++) bv[i] = bias[n0 + g * 4 + i];
  for (int p = pb; p < pe; p++) {
    __syncthreads();  // planes p-1..p+1 are staged; nobody reads plane p-2 any more
    if (p + 1 < pe) load(p + 2);
    f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
      for (int s = 0; s < 14; s++) {
        // both taps' offsets are the same for all lanes; tap 27 does not exist
        const int t0 = 2 * s, t1 = s == 13 ? 26 : 2 * s + 1;
        const int o0 = ((p + 3 + t0 / 9) & 3) * PL + t0 / 3 % 3 * HX + t0 % 3;
        const int o1 = ((p + 3 + t1 / 9) & 3) * PL + t1 / 3 % 3 * HX + t1 % 3;
        const int q = base + (odd ? o1 : o0) + c * 2 * MARCH_HV;
        uint4 b0 = ring[q], b1 = ring[q + step];
        if (s == 13 && odd) b0 = b1 = zero4;
        acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(w[c][s]), as_bf16x8(b0), acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(w[c][s]), as_bf16x8(b1), acc[1], 0, 0, 0);
      }
    if (p + 1 < pe) store(p + 2);
    // lane holds voxel r and channels g*4+i of each block
#pragma unroll
    for (int mb = 0; mb < 2; mb++) {
      const int m = mb ? m1 : m0, yy = y0 + (m >> ltx), xx = x0 + (m & (TX - 1));
      if (yy >= d1) continue;
      const size_t o = (size_t)(p * P + yy * d2 + xx) * Co + n0 + g * 4;
      uint2 mk = {0u, 0u};
      if (mask) mk = *(const uint2 *)(mask + o);
      bf16_t e[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        float val = acc[mb][i] + bv[i];
        if (relu) val = fmaxf(val, 0.f);
        const bf16_t k = (bf16_t)((i < 2 ? mk.x : mk.y) >> (16 * (i & 1)));
        if (mask && !bf_pos(k)) val = 0.f;
        e[i] = f2bf(val);
      }
      *(uint2 *)(out + o) =
          make_uint2(e[0] | ((uint32_t)e[1] << 16), e[2] | ((uint32_t)e[3] << 16));
    }
  }
}

// Forward of the one-channel stem (27 taps: one MFMA K-step, in k_conv3's order of taps):
// a workgroup stages STEM_SEG + 2 planes of a TY x TX tile (as k_conv3_march) with their
// halo at once and each lane gathers its 8 taps from there.  Gathered from memory with a
// bounds check per tap it took 456 us at 512 x 512 x 32.
constexpr int STEM_SEG = 32;

__global__ void __launch_bounds__(512) k_stem(const bf16_t *__restrict__ in,
                                              const bf16_t *__restrict__ W, int Kpad,
                                              const float *__restrict__ bias, int Co, int d0, int d1,
                                              int d2, int ltx, bf16_t *__restrict__ out) {
  __shared__ bf16_t pl[(STEM_SEG + 2) * MARCH_HV];
  const int TX = 1 << ltx, TY = 256 >> ltx, HX = TX + 2, HV = (TY + 2) * HX, P = d1 * d2;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int ntx = d2 >> ltx;
  const int x0 = (blockIdx.x % ntx) << ltx, y0 = blockIdx.x / ntx * TY;
  const int n0 = blockIdx.y * 16, pb = blockIdx.z * STEM_SEG, np = min(STEM_SEG, d0 - pb);
  if (tid < HV) {
    const int yy = y0 + tid / HX - 1, xx = x0 + tid % HX - 1;
    const bool ok = (unsigned)yy < (unsigned)d1 && (unsigned)xx < (unsigned)d2;
    for (int k = 0; k < np + 2; k++) {
      const int p = pb + k - 1;
      bf16_t e = 0;
      if (ok && (unsigned)p < (unsigned)d0) e = in[(size_t)p * P + yy * d2 + xx];
      pl[k * MARCH_HV + tid] = e;
    }
  }
  const bf16x8 w = as_bf16x8(*(const uint4 *)(W + (size_t)(n0 + r) * Kpad + g * 8));
  const int m0 = wave * 32 + r, m1 = m0 + 16;
  const int hv0 = (m0 >> ltx) * HX + (m0 & (TX - 1)), hv1 = (m1 >> ltx) * HX + (m1 & (TX - 1));
  int off[8];  // the lane's taps; those past the last (g = 3) are cleared below
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const int t = min(g * 8 + j, 26);
    off[j] = t / 9 * MARCH_HV + t / 3 % 3 * HX + t % 3;
  }
  float bv[4];
#pragma unroll
  for (int i = 0; i < 4; i++) bv[i] = bias[n0 + g * 4 + i];
  __syncthreads();
  for (int k = 0; k < np; k++)
#pragma unroll
    for (int mb = 0; mb < 2; mb++) {
      const int m = mb ? m1 : m0, yy = y0 + (m >> ltx), xx = x0 + (m & (TX - 1));
      const bf16_t *src = pl + k * MARCH_HV + (mb ? hv1 : hv0);
      uint32_t e[8];
#pragma unroll
      for (int j = 0; j < 8; j++) e[j] = src[off[j]];
      uint4 q = make_uint4(e[0] | e[1] << 16, e[2] | e[3] << 16, e[4] | e[5] << 16, e[6] | e[7] << 16);
      if (g == 3) q = make_uint4(q.x, q.y & 0xffffu, 0u, 0u);
      const f32x4 acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, as_bf16x8(q),
                                                                f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      if (yy >= d1) continue;
      bf16_t o[4];
#pragma unroll
      for (int i = 0; i < 4; i++) o[i] = f2bf(fmaxf(acc[i] + bv[i], 0.f));
      *(uint2 *)(out + (size_t)((pb + k) * P + yy * d2 + xx) * Co + n0 + g * 4) =
          make_uint2(o[0] | ((uint32_t)o[1] << 16), o[2] | ((uint32_t)o[3] << 16));
    }
}

// Weight gradient of a layer with Ci and Co multiples of 16: a workgroup takes 16 input
// and 16 output channels and all 27 taps, and walks over tiles of T0 x 8 x T2 voxels
// (T0 * T2 = WG_ROWS rows along d1, T2 = 1 << lt2).  A tile's gradients and its inputs
// with their halo are transposed on the way into LDS, so that a lane reads the 8 voxels
// of a row for its channel at once; the taps -1 and +1 along d1 are the same row shifted
// by one voxel, whose end comes from the halo words.  One read of inputs thus serves
// three taps and one of gradients serves 27; K of the product is 4 rows of 8 voxels, the
// 4 waves share the rows and the 27 tiles of sums stay in registers over all tiles.  The
// channel slots are rotated by row (XOR), so neither the transposed writes nor the reads
// collide in the banks.  The waves' sums are added in LDS and go to dW with one FP32
// atomic each.  Bound by staging and the matrix unit about equally.  A kernel with one
// wave per 16 x 64 outputs that gathered each operand from memory by 2-byte loads took
// 304 us a layer at 256 x 256 x 16 (mean of the 13 layers), this one 38 us.
constexpr int WG_ROWS = 64;

__device__ inline uint32_t wg_lo(uint32_t a, uint32_t b) { return (a & 0xffffu) | (b << 16); }
__device__ inline uint32_t wg_hi(uint32_t a, uint32_t b) { return (a >> 16) | (b & 0xffff0000u); }

// the 8 bf16 of q, by pairs
__device__ inline float wg_sum(uint4 q) {
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const uint32_t w = k == 0 ? q.x : k == 1 ? q.y : k == 2 ? q.z : q.w;
    s += __uint_as_float(w << 16) + __uint_as_float(w & 0xffff0000u);
  }
  return s;
}

// db[r] += the sums of the 16 lanes' channels over the workgroup; red: 64 floats
__device__ inline void wg_bias(float s, float *red, float *db) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  s += __shfl_xor(s, 16);
  s += __shfl_xor(s, 32);
  __syncthreads();  // red has been read
  if (lane < 16) red[wave * 16 + lane] = s;
  __syncthreads();
  if (threadIdx.x < 16)
    atomicAdd(db + lane, (red[lane] + red[16 + lane]) + (red[32 + lane] + red[48 + lane]));
}

__global__ void __launch_bounds__(256, 3) k_conv3_wgrad_tile(
    const bf16_t *__restrict__ in, int Ci, const bf16_t *__restrict__ gout, int Co, int d0, int d1,
    int d2, int lt2, int n1, int n2, int ntiles, float *__restrict__ dW, float *__restrict__ db) {
  extern __shared__ uint4 wg_smem[];
  const int T2 = 1 << lt2, T0 = WG_ROWS >> lt2, W2 = T2 + 2, NR = (T0 + 2) * W2;
  uint4 *gm = wg_smem;                       // [WG_ROWS][16] gradients
  uint4 *im = gm + WG_ROWS * 16;             // [NR][16] inputs
  uint32_t *ih = (uint32_t *)(im + NR * 16);  // [NR][16] the voxels before and after a row
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int co0 = blockIdx.y * 16, ci0 = blockIdx.z * 16;
  f32x4 acc[27];
#pragma unroll
  for (int t = 0; t < 27; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float bsum = 0.f;  // channel co0+r over the lane's voxels
  for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int o2 = (tile % n2) << lt2, o1 = tile / n2 % n1 * 8, o0 = tile / (n1 * n2) * T0;
    __syncthreads();  // the tile before has been read
    for (int u = tid; u < 2 * (WG_ROWS + NR); u += 256) {
      const bool grad = u < 2 * WG_ROWS;
      const int oct = u & 1, row = (grad ? u : u - 2 * WG_ROWS) >> 1;
      const int a0 = grad ? row >> lt2 : row / W2;
      const int q0 = o0 + (grad ? a0 : a0 - 1);
      const int q2 = o2 + (grad ? row & (T2 - 1) : row - a0 * W2 - 1);
      const bool ok = (unsigned)q0 < (unsigned)d0 && (unsigned)q2 < (unsigned)d2;
      const int C = grad ? Co : Ci;
      const bf16_t *src = (grad ? gout + co0 : in + ci0) + oct * 8;
      uint4 v[10];
#pragma unroll
      for (int j = 0; j < 10; j++) {
        const int q1 = o1 + j - 1;
        v[j] = make_uint4(0, 0, 0, 0);
        if (ok && (unsigned)q1 < (unsigned)d1 && (!grad || (j > 0 && j < 9)))
          v[j] = *(const uint4 *)(src + (((size_t)q0 * d1 + q1) * d2 + q2) * C);
      }
      uint4 *dst = (grad ? gm : im) + row * 16;
      uint32_t *dh = ih + row * 16;
#pragma unroll
      for (int k = 0; k < 4; k++) {
        uint32_t w[10];
#pragma unroll
        for (int j = 0; j < 10; j++) w[j] = k == 0 ? v[j].x : k == 1 ? v[j].y : k == 2 ? v[j].z : v[j].w;
        const int c = oct * 8 + 2 * k;
        dst[c ^ (row & 15)] = make_uint4(wg_lo(w[1], w[2]), wg_lo(w[3], w[4]), wg_lo(w[5], w[6]),
                                         wg_lo(w[7], w[8]));
        dst[(c + 1) ^ (row & 15)] = make_uint4(wg_hi(w[1], w[2]), wg_hi(w[3], w[4]),
                                               wg_hi(w[5], w[6]), wg_hi(w[7], w[8]));
        if (!grad) {
          dh[c ^ (row >> 2 & 15)] = wg_lo(w[0], w[9]);
          dh[(c + 1) ^ (row >> 2 & 15)] = wg_hi(w[0], w[9]);
        }
      }
    }
    __syncthreads();
#pragma unroll 1
    for (int ks = 0; ks < WG_ROWS / 16; ks++) {
      const int row = wave * (WG_ROWS / 4) + ks * 4 + g;
      const int a0 = row >> lt2, a2 = row & (T2 - 1);
      const uint4 gq = gm[row * 16 + (r ^ (row & 15))];
      if (ci0 == 0) bsum += wg_sum(gq);
      const bf16x8 a = as_bf16x8(gq);
#pragma unroll
      for (int e0 = 0; e0 < 3; e0++)
#pragma unroll
        for (int e2 = 0; e2 < 3; e2++) {
          const int hr = (a0 + e0) * W2 + a2 + e2;
          const uint4 m = im[hr * 16 + (r ^ (hr & 15))];
          const uint32_t h = ih[hr * 16 + (r ^ (hr >> 2 & 15))];
          const uint32_t s1 = (m.x >> 16) | (m.y << 16), s2 = (m.y >> 16) | (m.z << 16),
                         s3 = (m.z >> 16) | (m.w << 16);
          const int t = e0 * 9 + e2;
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a, as_bf16x8(make_uint4(wg_lo(h, m.x), s1, s2, s3)), acc[t], 0, 0, 0);
          acc[t + 3] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, as_bf16x8(m), acc[t + 3], 0, 0, 0);
          acc[t + 6] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a, as_bf16x8(make_uint4(s1, s2, s3, wg_hi(m.w, h))), acc[t + 6], 0, 0, 0);
        }
    }
  }
  // lane holds column ci0+r and rows co0+g*4+i
  float *red = (float *)wg_smem;  // [27][4][64]
  for (int w = 0; w < 4; w++) {
    __syncthreads();
    if (wave != w) continue;
#pragma unroll
    for (int t = 0; t < 27; t++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        float *q = red + (t * 4 + i) * 64 + lane;
        *q = w == 0 ? acc[t][i] : *q + acc[t][i];
      }
  }
  __syncthreads();
  for (int t = 0; t < 27; t++)
    atomicAdd(dW + (size_t)(co0 + g * 4 + wave) * 27 * Ci + (size_t)t * Ci + ci0 + r,
              red[(t * 4 + wave) * 64 + lane]);
  if (ci0 == 0) wg_bias(bsum, red, db + co0);
}

// Weight and bias gradient of the one-channel stem: k_conv3_wgrad_tile with the taps as
// the product's columns (two blocks of 16, 27 in use), each lane shifting its tap's row.
// Every operand gathered from memory by 2-byte loads took 465 us at 256 x 256 x 16, and
// the bias gradients of all layers another 290 us in kernels of their own.
__global__ void __launch_bounds__(256) k_stem_wgrad(const bf16_t *__restrict__ in,
                                                    const bf16_t *__restrict__ gout, int Co, int d0,
                                                    int d1, int d2, int lt2, int n1, int n2,
                                                    int ntiles, float *__restrict__ dW,
                                                    float *__restrict__ db) {
  extern __shared__ uint4 wg_smem[];
  const int T2 = 1 << lt2, T0 = WG_ROWS >> lt2, W2 = T2 + 2, NR = (T0 + 2) * W2;
  uint4 *gm = wg_smem;                // [WG_ROWS][16] gradients
  uint4 *im = gm + WG_ROWS * 16;      // [NR] inputs
  uint32_t *ih = (uint32_t *)(im + NR);  // [NR] the voxels before and after a row
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int co0 = blockIdx.y * 16;
  f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
  float bsum = 0.f;
  int trow[2], tsh[2];  // the column's tap: its row's offset and its shift along d1
#pragma unroll
  for (int nb = 0; nb < 2; nb++) {
    const int t = min(nb * 16 + r, 26);
    trow[nb] = t / 9 * W2 + t % 3;
    tsh[nb] = t / 3 % 3;
  }
  for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int o2 = (tile % n2) << lt2, o1 = tile / n2 % n1 * 8, o0 = tile / (n1 * n2) * T0;
    __syncthreads();  // the tile before has been read
    if (tid < 2 * WG_ROWS) {
      const int oct = tid & 1, row = tid >> 1;
      const int q0 = o0 + (row >> lt2), q2 = o2 + (row & (T2 - 1));
      uint4 v[8];
#pragma unroll
      for (int j = 0; j < 8; j++) {
        v[j] = make_uint4(0, 0, 0, 0);
        if (q0 < d0 && q2 < d2 && o1 + j < d1)
          v[j] = *(const uint4 *)(gout + (((size_t)q0 * d1 + o1 + j) * d2 + q2) * Co + co0 + oct * 8);
      }
#pragma unroll
      for (int k = 0; k < 4; k++) {
        uint32_t w[8];
#pragma unroll
        for (int j = 0; j < 8; j++) w[j] = k == 0 ? v[j].x : k == 1 ? v[j].y : k == 2 ? v[j].z : v[j].w;
        const int c = oct * 8 + 2 * k;
        gm[row * 16 + (c ^ (row & 15))] = make_uint4(wg_lo(w[0], w[1]), wg_lo(w[2], w[3]),
                                                     wg_lo(w[4], w[5]), wg_lo(w[6], w[7]));
        gm[row * 16 + ((c + 1) ^ (row & 15))] = make_uint4(wg_hi(w[0], w[1]), wg_hi(w[2], w[3]),
                                                           wg_hi(w[4], w[5]), wg_hi(w[6], w[7]));
      }
    }
    for (int row = 255 - tid; row < NR; row += 256) {  // from the waves without gradients on
      const int a0 = row / W2, q0 = o0 + a0 - 1, q2 = o2 + row - a0 * W2 - 1;
      const bool ok = (unsigned)q0 < (unsigned)d0 && (unsigned)q2 < (unsigned)d2;
      uint32_t e[10];
#pragma unroll
      for (int j = 0; j < 10; j++) {
        const int q1 = o1 + j - 1;
        e[j] = 0u;
        if (ok && (unsigned)q1 < (unsigned)d1) e[j] = in[((size_t)q0 * d1 + q1) * d2 + q2];
      }
      im[row] = make_uint4(e[1] | e[2] << 16, e[3] | e[4] << 16, e[5] | e[6] << 16, e[7] | e[8] << 16);
      ih[row] = e[0] | e[9] << 16;
    }
    __syncthreads();
    for (int ks = 0; ks < WG_ROWS / 16; ks++) {
      const int row = wave * (WG_ROWS / 4) + ks * 4 + g;
      const int hr = (row >> lt2) * W2 + (row & (T2 - 1));
      const uint4 gq = gm[row * 16 + (r ^ (row & 15))];
      bsum += wg_sum(gq);
#pragma unroll
      for (int nb = 0; nb < 2; nb++) {
        const uint4 m = im[hr + trow[nb]];
        const uint32_t h = ih[hr + trow[nb]];
        const uint32_t s1 = (m.x >> 16) | (m.y << 16), s2 = (m.y >> 16) | (m.z << 16),
                       s3 = (m.z >> 16) | (m.w << 16);
        uint4 b = m;
        if (tsh[nb] == 0) b = make_uint4(wg_lo(h, m.x), s1, s2, s3);
        if (tsh[nb] == 2) b = make_uint4(s1, s2, s3, wg_hi(m.w, h));
        acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(gq), as_bf16x8(b), acc[nb], 0, 0, 0);
      }
    }
  }
  // lane holds tap nb*16+r and rows co0+g*4+i
  float *red = (float *)wg_smem;  // [wave][2][4][64]
  __syncthreads();
#pragma unroll
  for (int nb = 0; nb < 2; nb++)
#pragma unroll
    for (int i = 0; i < 4; i++) red[((wave * 2 + nb) * 4 + i) * 64 + lane] = acc[nb][i];
  __syncthreads();
#pragma unroll
  for (int nb = 0; nb < 2; nb++) {
    float s = 0.f;
    for (int w = 0; w < 4; w++) s += red[((w * 2 + nb) * 4 + wave) * 64 + lane];
    if (nb * 16 + r < 27) atomicAdd(dW + (size_t)(co0 + g * 4 + wave) * 27 + nb * 16 + r, s);
  }
  wg_bias(bsum, red, db + co0);
}

// 2x2x2 average pool: fine dims (d0, d1, d2) -> coarse (d0/2, d1/2, d2/2); one
// thread per coarse voxel and 8 channels (C % 8 == 0), 16-byte loads and stores
__global__ void k_pool(const bf16_t *__restrict__ in, int C, int d0, int d1, int d2,
                       bf16_t *__restrict__ out) {
  const int e1 = d1 / 2, e2 = d2 / 2, C8 = C / 8;
  const size_t n = (size_t)(d0 / 2) * e1 * e2 * C8;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    const int c8 = (int)(i % C8);
    const int w = (int)(i / C8);  // coarse voxel (V < 2^31)
    const int q2 = w % e2, q1 = (w / e2) % e1, q0 = w / (e1 * e2);
    float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const size_t v = ((size_t)(2 * q0 + (k >> 2)) * d1 + (2 * q1 + ((k >> 1) & 1))) * d2 +
                       (2 * q2 + (k & 1));
      const uint4 q = *(const uint4 *)(in + v * C + 8 * c8);
      const uint32_t u[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int j = 0; j < 4; j++) {
        s[2 * j] += bf2f((bf16_t)(u[j] & 0xFFFFu));
        s[2 * j + 1] += bf2f((bf16_t)(u[j] >> 16));
      }
    }
    uint4 o;
    uint32_t *ou = (uint32_t *)&o;
#pragma unroll
    for (int j = 0; j < 4; j++)
      ou[j] = (uint32_t)f2bf(s[2 * j] * 0.125f) | ((uint32_t)f2bf(s[2 * j + 1] * 0.125f) << 16);
    *(uint4 *)(out + (size_t)w * C + 8 * c8) = o;
  }
}

// out[v] = [ low[parent(v)] (Ca channels) | skip[v] (Cb channels) ] on fine dims;
// one thread per 8 channels (Ca, Cb % 8 == 0), 16-byte copies
__global__ void k_upcat(const bf16_t *__restrict__ low, int Ca, const bf16_t *__restrict__ skip,
                        int Cb, int d0, int d1, int d2, bf16_t *__restrict__ out) {
  const int Ct8 = (Ca + Cb) / 8, Ca8 = Ca / 8;
  const size_t n = (size_t)d0 * d1 * d2 * Ct8;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    const int c8 = (int)(i % Ct8);
    const int v = (int)(i / Ct8);  // V < 2^31
    uint4 q;
    if (c8 < Ca8) {
      const int p2 = v % d2, p1 = (v / d2) % d1, p0 = v / (d1 * d2);
      const size_t u = ((size_t)(p0 / 2) * (d1 / 2) + p1 / 2) * (d2 / 2) + p2 / 2;
      q = *(const uint4 *)(low + u * Ca + 8 * c8);
    } else {
      q = *(const uint4 *)(skip + (size_t)v * Cb + 8 * (c8 - Ca8));
    }
    *(uint4 *)(out + i * 8) = q;
  }
}

// glow[u][c] = sum over the 8 children v of u of gcat[v][c], c < Ca (coarse dims)
__global__ void k_up_bwd(const bf16_t *__restrict__ gcat, int Ca, int Ct, int e0, int e1, int e2,
                         bf16_t *__restrict__ glow) {
  const size_t n = (size_t)e0 * e1 * e2 * Ca;
  const int d1 = 2 * e1, d2 = 2 * e2;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    const int c = (int)(i % Ca);
    const size_t w = i / Ca;
    const int q2 = (int)(w % e2), q1 = (int)((w / e2) % e1), q0 = (int)(w / ((size_t)e1 * e2));
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const size_t v = ((size_t)(2 * q0 + (k >> 2)) * d1 + (2 * q1 + ((k >> 1) & 1))) * d2 +
                       (2 * q2 + (k & 1));
      s += bf2f(gcat[v * Ct + c]);
    }
    glow[i] = f2bf(s);
  }
}

// ge[v][c] = gcat[v][Ca+c] + [e[v][c] > 0] * gpool[parent(v)][c] / 8 (fine dims);
// gcat's skip part is already masked by the concatenated activation.
__global__ void k_skip_bwd(const bf16_t *__restrict__ gcat, int Ca, int Ct,
                           const bf16_t *__restrict__ gpool, const bf16_t *__restrict__ e, int Cb,
                           int d0, int d1, int d2, bf16_t *__restrict__ ge) {
  const size_t n = (size_t)d0 * d1 * d2 * Cb;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    const int c = (int)(i % Cb);
    const size_t v = i / Cb;
    const int p2 = (int)(v % d2), p1 = (int)((v / d2) % d1), p0 = (int)(v / ((size_t)d1 * d2));
    const size_t u = ((size_t)(p0 / 2) * (d1 / 2) + p1 / 2) * (d2 / 2) + p2 / 2;
    float s = bf2f(gcat[v * Ct + Ca + c]);
    if (bf_pos(e[i])) s += bf2f(gpool[u * Cb + c]) * 0.125f;
    ge[i] = f2bf(s);
  }
}

// network input: t[v] = bf16(x[v] * scale)
__global__ void k_prep(const float *__restrict__ x, float scale, size_t n, bf16_t *__restrict__ t) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    t[i] = f2bf(x[i] * scale);
}

// head: out[v] = (x[v]*scale + sum_c d[v][c]*wh[c] + bh) / scale
__global__ void k_head_fwd(const bf16_t *__restrict__ d, int C, const float *__restrict__ wh,
                           const float *__restrict__ bh, const float *x, float scale, size_t n,
                           float *out) {
  // C == 16: two 16-byte loads per voxel
  for (size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x; v < n;
       v += (size_t)gridDim.x * blockDim.x) {
    const uint4 q0 = *(const uint4 *)(d + v * C), q1 = *(const uint4 *)(d + v * C + 8);
    const uint32_t u[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
    float h = bh[0];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      h += bf2f((bf16_t)(u[j] & 0xFFFFu)) * wh[2 * j];
      h += bf2f((bf16_t)(u[j] >> 16)) * wh[2 * j + 1];
    }
    out[v] = (x[v] * scale + h) / scale;
  }
}

// head backward and the loss mean((x*s + h - t*s)^2):
// g = 2 res / n; loss += res^2 / n; dwh[c] += g d[v][c]; dbh += g;
// gd[v][c] = bf16(g wh[c]) [d[v][c] > 0].  Block size 256, C <= 16.
__global__ void __launch_bounds__(256) k_head_bwd(const bf16_t *__restrict__ d, int C,
                                                  const float *__restrict__ wh,
                                                  const float *__restrict__ bh,
                                                  const float *__restrict__ x,
                                                  const float *__restrict__ tgt, float scale,
                                                  size_t n, double *loss, float *dwh, float *dbh,
                                                  bf16_t *__restrict__ gd) {
  __shared__ float red[17][256];
  __shared__ double redl[256];
  const int t = threadIdx.x;
  float sw[16] = {0.f}, sb = 0.f;
  double sl = 0.0;
  const float inv_n = 1.f / (float)n;
  for (size_t v = (size_t)blockIdx.x * blockDim.x + t; v < n; v += (size_t)gridDim.x * blockDim.x) {
    float h = bh[0];
    float dv[16];
    for (int c = 0; c < C; c++) {
      dv[c] = bf2f(d[v * C + c]);
      h += dv[c] * wh[c];
    }
    const float res = x[v] * scale + h - tgt[v] * scale;
    const float gv = 2.f * res * inv_n;
    sl += (double)res * res;
    sb += gv;
    for (int c = 0; c < C; c++) {
      sw[c] += gv * dv[c];
      gd[v * C + c] = dv[c] > 0.f ? f2bf(gv * wh[c]) : (bf16_t)0;
    }
  }
  for (int c = 0; c < C; c++) red[c][t] = sw[c];
  red[16][t] = sb;
  redl[t] = sl;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (t < s) {
      for (int c = 0; c < C; c++) red[c][t] += red[c][t + s];
      red[16][t] += red[16][t + s];
      redl[t] += redl[t + s];
    }
    __syncthreads();
  }
  if (t < C) atomicAdd(dwh + t, red[t][0]);
  if (t == 0) {
    atomicAdd(dbh, red[16][0]);
    atomicAdd(loss, redl[0] / (double)n);
  }
}

// bf16 weight layouts from the FP32 master [Co][27*Ci]:
//   forward  Wf[co][kk], kk = tap*Ci + ci < Kpad (zero beyond 27*Ci)
//   backward Wb[ci][kk'], kk' = tap'*Co + co < Kpadb, Wb = W[co][(26-tap')*Ci + ci]
__global__ void k_wprep(const float *__restrict__ w, int Ci, int Co, int Kpad, int Kpadb,
                        bf16_t *__restrict__ Wf, bf16_t *__restrict__ Wb) {
  const size_t nf = (size_t)Co * Kpad, nb = (size_t)Ci * Kpadb;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < nf + nb;
       i += (size_t)gridDim.x * blockDim.x) {
    if (i < nf) {
      const int co = (int)(i / Kpad), kk = (int)(i % Kpad);
      Wf[i] = kk < 27 * Ci ? f2bf(w[(size_t)co * 27 * Ci + kk]) : (bf16_t)0;
    } else {
      const size_t j = i - nf;
      const int ci = (int)(j / Kpadb), kk = (int)(j % Kpadb);
      bf16_t val = 0;
      if (kk < 27 * Co) {
        const int tp = kk / Co, co = kk % Co;
        val = f2bf(w[(size_t)co * 27 * Ci + (26 - tp) * Ci + ci]);
      }
      Wb[j] = val;
    }
  }
}

__global__ void k_adam(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                       float *__restrict__ v, size_t n, float lr, float b1, float b2, float eps,
                       float bc1, float bc2) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
  }
}

__global__ void k_fill(float *__restrict__ p, size_t n, float val) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = val;
}

__global__ void k_fill_d(double *p, double val) { *p = val; }

// ---------------------------------------------------------------------------
// host side
namespace {

constexpr int NCONV = 14;
// (level, C_in, C_out) of each 3x3x3 conv with base channels 16
const int kConvSpec[NCONV][3] = {{0, 1, 16},   {0, 16, 16},  {1, 16, 32}, {1, 32, 32},
                                 {2, 32, 64},  {2, 64, 64},  {3, 64, 128}, {3, 128, 128},
                                 {2, 192, 64}, {2, 64, 64},  {1, 96, 32}, {1, 32, 32},
                                 {0, 48, 16},  {0, 16, 16}};
constexpr int HEAD_C = 16;

struct Conv {
  int lvl, Ci, Co, Kpad, Kpadb;
  size_t w_off, b_off;  // into the parameter vector
  bf16_t *Wf = nullptr, *Wb = nullptr;
};

int grid1(size_t n) { return (int)std::min<size_t>((n + 255) / 256, 8192); }

}  // namespace

struct xt_unet {
  int dev = 0;
  hipStream_t st = nullptr;  // the stream of the synchronous entry points
  int dims[4][3];
  size_t V[4];
  float scale = 1.f;
  bool train = false;
  Conv conv[NCONV];
  size_t head_w = 0, head_b = 0;
  int64_t nparam = 0;
  float *params = nullptr, *grads = nullptr, *adam_m = nullptr, *adam_v = nullptr;
  int64_t adam_t = 0;
  bool wdirty = true;
  bf16_t *wbuf = nullptr;
  // activations
  bf16_t *t_in, *e1a, *e1, *p1, *e2a, *e2, *p2, *e3a, *e3, *p3, *ba, *bb, *u3, *d3a, *d3, *u2,
      *d2a, *d2, *u1, *d1a, *d1;
  // activation gradients (train)
  bf16_t *g_d1, *g_d1a, *g_u1, *g_d2, *g_d2a, *g_u2, *g_d3, *g_d3a, *g_u3, *g_bb, *g_ba, *g_p3,
      *g_e3, *g_e3a, *g_p2, *g_e2, *g_e2a, *g_p1, *g_e1, *g_e1a;
  bf16_t *abuf = nullptr, *gbuf = nullptr;
  double *loss_dev = nullptr;
  float *stage = nullptr;  // [2][V0] host-call staging (input, target/output)
  hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
  double fwd_ms = 0, bwd_ms = 0;
};

namespace {

// carve `count` bf16 elements (16-byte aligned) from a running offset
struct Carver {
  size_t off = 0;
  std::vector<std::pair<bf16_t **, size_t>> items;
  void add(bf16_t **p, size_t count) {
    items.push_back({p, off});
    off += (count + 127) / 128 * 128;
  }
  void assign(bf16_t *base) {
    for (auto &it : items) *it.first = base + it.second;
  }
};

int pow2_divisor(int n, int cap) {  // largest power of two dividing n, at most cap
  int p = 1;
  while (p * 2 <= cap && n % (p * 2) == 0) p *= 2;
  return p;
}

// dynamic LDS of k_conv3_march: four planes
size_t march_lds(int Ci) { return (size_t)4 * (Ci / 8) * MARCH_HV * sizeof(uint4); }

void launch_conv(xt_unet *u, hipStream_t st, const bf16_t *in, int Ci, const bf16_t *W, int Kpad,
                 const float *bias, int Co, const int *d, bf16_t *out, int relu,
                 const bf16_t *mask) {
  const int V = d[0] * d[1] * d[2];
  const int NB = (Co % 64 == 0) ? 4 : (Co % 32 == 0) ? 2 : 1;
  if ((Ci == 16 || Ci == 48) && Co % 16 == 0 && d[2] % 8 == 0) {
    // a workgroup (16 channels) or two thirds of one (48) a CU over two rounds, but 8
    // planes at least: a segment stages two more than it computes
    const int TX = pow2_divisor(d[2], 32), ltx = __builtin_ctz(TX), TY = 256 / TX;
    const int nt = (d[2] / TX) * ((d[1] + TY - 1) / TY) * (Co / 16);
    const int nseg = std::max(1, std::min((Ci == 16 ? 1536 : 512) / nt, d[0] / 8));
    const int seg = (d[0] + nseg - 1) / nseg;
    const dim3 grid((d[2] / TX) * ((d[1] + TY - 1) / TY), Co / 16, (d[0] + seg - 1) / seg);
    const size_t lds = march_lds(Ci);
    if (Ci == 16)
      hipLaunchKernelGGL((k_conv3_march<1>), grid, dim3(512), lds, st, in, W, Kpad, bias, Co, d[0],
                         d[1], d[2], ltx, seg, out, relu, mask);
    else
      hipLaunchKernelGGL((k_conv3_march<3>), grid, dim3(512), lds, st, in, W, Kpad, bias, Co, d[0],
                         d[1], d[2], ltx, seg, out, relu, mask);
    return;
  }
  if (Ci % 32 == 0) {
    const int TX = pow2_divisor(d[2], 32), TY = pow2_divisor(d[1], 128 / TX);
    const size_t lds = (size_t)3 * (TY + 2) * (TX + 2) * (32 + 8) * sizeof(bf16_t);
    dim3 grid(d[0] * (d[1] / TY) * (d[2] / TX), Co / (16 * NB));
#define UN_LDS(NB_)                                                                                \
  hipLaunchKernelGGL((k_conv3_lds<2, NB_>), grid, dim3(256), lds, st, in, Ci, W, Kpad, bias, Co,   \
                     d[0], d[1], d[2], TY, TX, out, relu, mask)
    if (NB == 1) UN_LDS(1);
    else if (NB == 2) UN_LDS(2);
    else UN_LDS(4);
#undef UN_LDS
    return;
  }
  // 16 -> 32 channels at half resolution where d2 has no factor 8
  hipLaunchKernelGGL((k_conv3<4, 2>), dim3((V + 255) / 256, Co / 32), dim3(256), 0, st, in, Ci, W,
                     Kpad, bias, Co, d[0], d[1], d[2], out, relu, mask);
}

// forward of the stem: + bias, ReLU
void launch_stem(hipStream_t st, const bf16_t *in, const bf16_t *W, int Kpad, const float *bias,
                 int Co, const int *d, bf16_t *out) {
  const int TX = pow2_divisor(d[2], 32), TY = 256 / TX;
  hipLaunchKernelGGL(k_stem, dim3((d[2] / TX) * ((d[1] + TY - 1) / TY), Co / 16,
                                  (d[0] + STEM_SEG - 1) / STEM_SEG),
                     dim3(512), 0, st, in, W, Kpad, bias, Co, d[0], d[1], d[2], __builtin_ctz(TX), out);
}

// dW and db of a layer with 1 (the stem) or 16 * n input channels
void launch_wgrad(hipStream_t st, const bf16_t *in, int Ci, const bf16_t *gout, int Co,
                  const int *d, float *dW, float *db) {
  // rows of 8 voxels along d1 in tiles of 8 (or 4, where d2 is less) along d2; as many
  // workgroups as run at once (3 a CU by their LDS), each over the same number of tiles
  const int lt2 = d[2] >= 8 ? 3 : 2, T2 = 1 << lt2, T0 = WG_ROWS >> lt2;
  const int n2 = (d[2] + T2 - 1) / T2, n1 = (d[1] + 7) / 8, n0 = (d[0] + T0 - 1) / T0;
  const int ntiles = n0 * n1 * n2, cb = Ci == 1 ? 1 : Ci / 16;
  const int nx = std::max(1, 768 / (cb * (Co / 16))), per = (ntiles + nx - 1) / nx;
  const dim3 grid((ntiles + per - 1) / per, Co / 16, cb);
  const size_t grad = (size_t)WG_ROWS * 16 * sizeof(uint4);
  const size_t rows = (size_t)(T0 + 2) * (T2 + 2) * (sizeof(uint4) + sizeof(uint32_t));
  if (Ci == 1)
    hipLaunchKernelGGL(k_stem_wgrad, grid, dim3(256), grad + rows, st, in, gout, Co, d[0], d[1], d[2],
                       lt2, n1, n2, ntiles, dW, db);
  else
    hipLaunchKernelGGL(k_conv3_wgrad_tile, grid, dim3(256), grad + 16 * rows, st, in, Ci, gout, Co,
                       d[0], d[1], d[2], lt2, n1, n2, ntiles, dW, db);
}

// forward of every layer on stream st; x is the float32 input volume
void enqueue_forward(xt_unet *u, const float *x, float *out, hipStream_t st) {
  if (u->wdirty) {
    for (int l = 0; l < NCONV; l++) {
      const Conv &c = u->conv[l];
      const size_t n = (size_t)c.Co * c.Kpad + (size_t)c.Ci * c.Kpadb;
      hipLaunchKernelGGL(k_wprep, dim3(grid1(n)), dim3(256), 0, st, u->params + c.w_off, c.Ci,
                         c.Co, c.Kpad, c.Kpadb, c.Wf, c.Wb);
    }
    u->wdirty = false;
  }
  const size_t V0 = u->V[0];
  hipLaunchKernelGGL(k_prep, dim3(grid1(V0)), dim3(256), 0, st, x, u->scale, V0, u->t_in);
  auto conv = [&](int l, const bf16_t *in, bf16_t *o) {
    const Conv &c = u->conv[l];
    launch_conv(u, st, in, c.Ci, c.Wf, c.Kpad, u->params + c.b_off, c.Co, u->dims[c.lvl], o, 1,
                nullptr);
  };
  auto pool = [&](int lvl, const bf16_t *in, int C, bf16_t *o) {
    const int *d = u->dims[lvl];
    hipLaunchKernelGGL(k_pool, dim3(grid1(u->V[lvl + 1] * C / 8)), dim3(256), 0, st, in, C, d[0],
                       d[1], d[2], o);
  };
  auto upcat = [&](int lvl, const bf16_t *low, int Ca, const bf16_t *skip, int Cb, bf16_t *o) {
    const int *d = u->dims[lvl];
    hipLaunchKernelGGL(k_upcat, dim3(grid1(u->V[lvl] * (Ca + Cb) / 8)), dim3(256), 0, st, low, Ca,
                       skip, Cb, d[0], d[1], d[2], o);
  };
  launch_stem(st, u->t_in, u->conv[0].Wf, u->conv[0].Kpad, u->params + u->conv[0].b_off, u->conv[0].Co,
              u->dims[0], u->e1a);
  conv(1, u->e1a, u->e1);
  pool(0, u->e1, 16, u->p1);
  conv(2, u->p1, u->e2a);
  conv(3, u->e2a, u->e2);
  pool(1, u->e2, 32, u->p2);
  conv(4, u->p2, u->e3a);
  conv(5, u->e3a, u->e3);
  pool(2, u->e3, 64, u->p3);
  conv(6, u->p3, u->ba);
  conv(7, u->ba, u->bb);
  upcat(2, u->bb, 128, u->e3, 64, u->u3);
  conv(8, u->u3, u->d3a);
  conv(9, u->d3a, u->d3);
  upcat(1, u->d3, 64, u->e2, 32, u->u2);
  conv(10, u->u2, u->d2a);
  conv(11, u->d2a, u->d2);
  upcat(0, u->d2, 32, u->e1, 16, u->u1);
  conv(12, u->u1, u->d1a);
  conv(13, u->d1a, u->d1);
  if (out)  // training recomputes the head inside its backward
    hipLaunchKernelGGL(k_head_fwd, dim3(grid1(V0)), dim3(256), 0, st, u->d1, HEAD_C,
                       u->params + u->head_w, u->params + u->head_b, x, u->scale, V0, out);
}

// backward after enqueue_forward(x): gradient of mean((out - tgt)^2 * scale^2)
void enqueue_backward(xt_unet *u, const float *x, const float *tgt, hipStream_t st) {
  const size_t V0 = u->V[0];
  hipLaunchKernelGGL(k_fill, dim3(grid1(u->nparam)), dim3(256), 0, st, u->grads,
                     (size_t)u->nparam, 0.f);
  hipLaunchKernelGGL(k_fill_d, dim3(1), dim3(1), 0, st, u->loss_dev, 0.0);
  hipLaunchKernelGGL(k_head_bwd, dim3(std::min<size_t>((V0 + 255) / 256, 1024)), dim3(256), 0, st,
                     u->d1, HEAD_C, u->params + u->head_w, u->params + u->head_b, x, tgt, u->scale,
                     V0, u->loss_dev, u->grads + u->head_w, u->grads + u->head_b, u->g_d1);
  // conv l: input `in`, pre-activation gradient `g`; input gradient to `gin`
  // (masked by `in` when it is a ReLU output), skipped for the stem
  auto back = [&](int l, const bf16_t *in, const bf16_t *g, bf16_t *gin, bool in_relu) {
    const Conv &c = u->conv[l];
    const int *d = u->dims[c.lvl];
    launch_wgrad(st, in, c.Ci, g, c.Co, d, u->grads + c.w_off, u->grads + c.b_off);
    if (gin)
      launch_conv(u, st, g, c.Co, c.Wb, c.Kpadb, nullptr, c.Ci, d, gin, 0, in_relu ? in : nullptr);
  };
  auto up_bwd = [&](int lvl_coarse, const bf16_t *gcat, int Ca, int Ct, bf16_t *glow) {
    const int *e = u->dims[lvl_coarse];
    hipLaunchKernelGGL(k_up_bwd, dim3(grid1(u->V[lvl_coarse] * Ca)), dim3(256), 0, st, gcat, Ca,
                       Ct, e[0], e[1], e[2], glow);
  };
  auto skip_bwd = [&](int lvl, const bf16_t *gcat, int Ca, int Ct, const bf16_t *gpool,
                      const bf16_t *e, int Cb, bf16_t *ge) {
    const int *d = u->dims[lvl];
    hipLaunchKernelGGL(k_skip_bwd, dim3(grid1(u->V[lvl] * Cb)), dim3(256), 0, st, gcat, Ca, Ct,
                       gpool, e, Cb, d[0], d[1], d[2], ge);
  };
  back(13, u->d1a, u->g_d1, u->g_d1a, true);
  back(12, u->u1, u->g_d1a, u->g_u1, true);
  up_bwd(1, u->g_u1, 32, 48, u->g_d2);
  back(11, u->d2a, u->g_d2, u->g_d2a, true);
  back(10, u->u2, u->g_d2a, u->g_u2, true);
  up_bwd(2, u->g_u2, 64, 96, u->g_d3);
  back(9, u->d3a, u->g_d3, u->g_d3a, true);
  back(8, u->u3, u->g_d3a, u->g_u3, true);
  up_bwd(3, u->g_u3, 128, 192, u->g_bb);
  back(7, u->ba, u->g_bb, u->g_ba, true);
  back(6, u->p3, u->g_ba, u->g_p3, false);
  skip_bwd(2, u->g_u3, 128, 192, u->g_p3, u->e3, 64, u->g_e3);
  back(5, u->e3a, u->g_e3, u->g_e3a, true);
  back(4, u->p2, u->g_e3a, u->g_p2, false);
  skip_bwd(1, u->g_u2, 64, 96, u->g_p2, u->e2, 32, u->g_e2);
  back(3, u->e2a, u->g_e2, u->g_e2a, true);
  back(2, u->p1, u->g_e2a, u->g_p1, false);
  skip_bwd(0, u->g_u1, 32, 48, u->g_p1, u->e1, 16, u->g_e1);
  back(1, u->e1a, u->g_e1, u->g_e1a, true);
  back(0, u->t_in, u->g_e1a, nullptr, false);
}

void free_net(xt_unet *u) {
  if (!u) return;
  void *bufs[] = {u->params, u->grads, u->adam_m, u->adam_v, u->wbuf,
                  u->abuf,   u->gbuf,  u->loss_dev, u->stage};
  for (void *b : bufs)
    if (b) (void)hipFree(b);
  for (hipEvent_t e : u->ev)
    if (e) (void)hipEventDestroy(e);
  if (u->st) (void)hipStreamDestroy(u->st);
  delete u;
}

}  // namespace

void xt_unet_shape(const xt_unet *u, int *d0, int *d1, int *d2) {
  *d0 = u->dims[0][0];
  *d1 = u->dims[0][1];
  *d2 = u->dims[0][2];
}

int xt_unet_forward_on(xt_unet *u, const float *in, float *out, hipStream_t st) {
  enqueue_forward(u, in, out, st);
  UN_HIP(hipGetLastError());
  return XT_OK;
}

extern "C" int xt_unet_create(int32_t d0, int32_t d1, int32_t d2, float scale, uint64_t seed,
                              int32_t train, xt_unet **net) {
  if (!net) return xt_report_error(XT_E_ARG, "null net pointer");
  *net = nullptr;
  if (d0 <= 0 || d1 <= 0 || d2 <= 0 || d0 % 8 || d1 % 8 || d2 % 8)
    return xt_report_error(XT_E_ARG, "U-Net volume %dx%dx%d: each size must be a positive "
                           "multiple of 8", d0, d1, d2);
  if ((int64_t)d0 * d1 * d2 * 192 >= (int64_t)1 << 31)
    return xt_report_error(XT_E_ARG, "U-Net volume %dx%dx%d too large (V*192 must be < 2^31)",
                           d0, d1, d2);
  if (!(scale > 0.f) || !std::isfinite(scale))
    return xt_report_error(XT_E_ARG, "U-Net input scale must be positive");
  xt_unet *u = new xt_unet();
  u->scale = scale;
  u->train = train != 0;
  (void)hipGetDevice(&u->dev);
  for (int l = 0; l < 4; l++) {
    u->dims[l][0] = d0 >> l;
    u->dims[l][1] = d1 >> l;
    u->dims[l][2] = d2 >> l;
    u->V[l] = (size_t)u->dims[l][0] * u->dims[l][1] * u->dims[l][2];
  }
  // parameters
  size_t off = 0, wcount = 0;
  for (int l = 0; l < NCONV; l++) {
    Conv &c = u->conv[l];
    c.lvl = kConvSpec[l][0];
    c.Ci = kConvSpec[l][1];
    c.Co = kConvSpec[l][2];
    c.Kpad = (27 * c.Ci + 31) / 32 * 32;
    c.Kpadb = (27 * c.Co + 31) / 32 * 32;
    c.w_off = off;
    off += (size_t)c.Co * 27 * c.Ci;
    c.b_off = off;
    off += c.Co;
    wcount += (size_t)c.Co * c.Kpad + (size_t)c.Ci * c.Kpadb;
  }
  u->head_w = off;
  off += HEAD_C;
  u->head_b = off;
  off += 1;
  u->nparam = (int64_t)off;
  auto fail = [&](int rc) {
    free_net(u);
    return rc;
  };
#define UN_ALLOC(ptr, bytes)                                                               \
  do {                                                                                     \
    hipError_t _e = hipMalloc((void **)&(ptr), (bytes));                                   \
    if (_e != hipSuccess)                                                                  \
      return fail(xt_report_error(XT_E_HIP, "U-Net allocation of %zu bytes: %s",           \
                                  (size_t)(bytes), hipGetErrorString(_e)));                \
  } while (0)
  {
    const hipError_t e = hipFuncSetAttribute((const void *)k_conv3_march<3>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)march_lds(48));
    if (e != hipSuccess)
      return fail(xt_report_error(XT_E_HIP, "U-Net: %zu bytes of LDS: %s", march_lds(48),
                                  hipGetErrorString(e)));
  }
  UN_ALLOC(u->params, off * sizeof(float));
  UN_ALLOC(u->wbuf, wcount * sizeof(bf16_t) + 256);
  {
    size_t w = 0;
    for (int l = 0; l < NCONV; l++) {
      Conv &c = u->conv[l];
      c.Wf = u->wbuf + w;
      w += (size_t)c.Co * c.Kpad;
      c.Wb = u->wbuf + w;
      w += (size_t)c.Ci * c.Kpadb;
    }
  }
  const size_t *V = u->V;
  Carver a;
  a.add(&u->t_in, V[0]);
  a.add(&u->e1a, V[0] * 16);
  a.add(&u->e1, V[0] * 16);
  a.add(&u->p1, V[1] * 16);
  a.add(&u->e2a, V[1] * 32);
  a.add(&u->e2, V[1] * 32);
  a.add(&u->p2, V[2] * 32);
  a.add(&u->e3a, V[2] * 64);
  a.add(&u->e3, V[2] * 64);
  a.add(&u->p3, V[3] * 64);
  a.add(&u->ba, V[3] * 128);
  a.add(&u->bb, V[3] * 128);
  a.add(&u->u3, V[2] * 192);
  a.add(&u->d3a, V[2] * 64);
  a.add(&u->d3, V[2] * 64);
  a.add(&u->u2, V[1] * 96);
  a.add(&u->d2a, V[1] * 32);
  a.add(&u->d2, V[1] * 32);
  a.add(&u->u1, V[0] * 48);
  a.add(&u->d1a, V[0] * 16);
  a.add(&u->d1, V[0] * 16);
  UN_ALLOC(u->abuf, a.off * sizeof(bf16_t));
  a.assign(u->abuf);
  if (u->train) {
    Carver gc;
    gc.add(&u->g_d1, V[0] * 16);
    gc.add(&u->g_d1a, V[0] * 16);
    gc.add(&u->g_u1, V[0] * 48);
    gc.add(&u->g_d2, V[1] * 32);
    gc.add(&u->g_d2a, V[1] * 32);
    gc.add(&u->g_u2, V[1] * 96);
    gc.add(&u->g_d3, V[2] * 64);
    gc.add(&u->g_d3a, V[2] * 64);
    gc.add(&u->g_u3, V[2] * 192);
    gc.add(&u->g_bb, V[3] * 128);
    gc.add(&u->g_ba, V[3] * 128);
    gc.add(&u->g_p3, V[3] * 64);
    gc.add(&u->g_e3, V[2] * 64);
    gc.add(&u->g_e3a, V[2] * 64);
    gc.add(&u->g_p2, V[2] * 32);
    gc.add(&u->g_e2, V[1] * 32);
    gc.add(&u->g_e2a, V[1] * 32);
    gc.add(&u->g_p1, V[1] * 16);
    gc.add(&u->g_e1, V[0] * 16);
    gc.add(&u->g_e1a, V[0] * 16);
    UN_ALLOC(u->gbuf, gc.off * sizeof(bf16_t));
    gc.assign(u->gbuf);
    UN_ALLOC(u->grads, off * sizeof(float));
    UN_ALLOC(u->adam_m, off * sizeof(float));
    UN_ALLOC(u->adam_v, off * sizeof(float));
    UN_ALLOC(u->loss_dev, sizeof(double));
  }
#undef UN_ALLOC
  if (hipStreamCreate(&u->st) != hipSuccess) return fail(xt_report_error(XT_E_HIP, "stream"));
  for (auto &e : u->ev)
    if (hipEventCreate(&e) != hipSuccess) return fail(xt_report_error(XT_E_HIP, "events"));
  // He-normal weights, zero biases, zero head
  std::vector<float> h(off, 0.f);
  std::mt19937_64 rng(seed);
  for (int l = 0; l < NCONV; l++) {
    const Conv &c = u->conv[l];
    std::normal_distribution<float> nd(0.f, std::sqrt(2.f / (27.f * c.Ci)));
    for (size_t i = 0; i < (size_t)c.Co * 27 * c.Ci; i++) h[c.w_off + i] = nd(rng);
  }
  int rc = xt_unet_set_params(u, h.data(), (int64_t)off);
  if (rc != XT_OK) return fail(rc);
  *net = u;
  return XT_OK;
}

extern "C" void xt_unet_destroy(xt_unet *u) { free_net(u); }

extern "C" int64_t xt_unet_param_count(const xt_unet *u) { return u ? u->nparam : 0; }

extern "C" int xt_unet_get_scale(const xt_unet *u, float *scale) {
  if (!u || !scale) return xt_report_error(XT_E_ARG, "null argument");
  *scale = u->scale;
  return XT_OK;
}

extern "C" int xt_unet_get_params(xt_unet *u, float *host, int64_t n) {
  if (!u || !host || n != u->nparam)
    return xt_report_error(XT_E_ARG, "get_params: need %lld floats", (long long)(u ? u->nparam : 0));
  UN_HIP(hipStreamSynchronize(u->st));
  UN_HIP(hipMemcpy(host, u->params, n * sizeof(float), hipMemcpyDeviceToHost));
  return XT_OK;
}

extern "C" int xt_unet_set_params(xt_unet *u, const float *host, int64_t n) {
  if (!u || !host || n != u->nparam)
    return xt_report_error(XT_E_ARG, "set_params: need %lld floats", (long long)(u ? u->nparam : 0));
  UN_HIP(hipStreamSynchronize(u->st));
  UN_HIP(hipMemcpy(u->params, host, n * sizeof(float), hipMemcpyHostToDevice));
  if (u->train) {
    hipLaunchKernelGGL(k_fill, dim3(grid1(n)), dim3(256), 0, u->st, u->adam_m, (size_t)n, 0.f);
    hipLaunchKernelGGL(k_fill, dim3(grid1(n)), dim3(256), 0, u->st, u->adam_v, (size_t)n, 0.f);
    hipLaunchKernelGGL(k_fill, dim3(grid1(n)), dim3(256), 0, u->st, u->grads, (size_t)n, 0.f);
    u->adam_t = 0;
  }
  u->wdirty = true;
  UN_HIP(hipStreamSynchronize(u->st));
  return XT_OK;
}

extern "C" int xt_unet_forward(xt_unet *u, const float *in, float *out) {
  if (!u || !in || !out) return xt_report_error(XT_E_ARG, "null argument");
  UN_HIP(hipEventRecord(u->ev[0], u->st));
  UN_TRY(xt_unet_forward_on(u, in, out, u->st));
  UN_HIP(hipEventRecord(u->ev[1], u->st));
  UN_HIP(hipEventSynchronize(u->ev[1]));
  float ms = 0.f;
  UN_HIP(hipEventElapsedTime(&ms, u->ev[0], u->ev[1]));
  u->fwd_ms = ms;
  return XT_OK;
}

extern "C" int xt_unet_loss_grad(xt_unet *u, const float *in, const float *tgt, double *loss,
                                 float *grad_host) {
  if (!u || !in || !tgt) return xt_report_error(XT_E_ARG, "null argument");
  if (!u->train) return xt_report_error(XT_E_ARG, "network was created without training buffers");
  UN_HIP(hipEventRecord(u->ev[0], u->st));
  enqueue_forward(u, in, nullptr, u->st);
  UN_HIP(hipEventRecord(u->ev[1], u->st));
  enqueue_backward(u, in, tgt, u->st);
  UN_HIP(hipGetLastError());
  UN_HIP(hipEventRecord(u->ev[2], u->st));
  UN_HIP(hipEventSynchronize(u->ev[2]));
  float f = 0.f, b = 0.f;
  UN_HIP(hipEventElapsedTime(&f, u->ev[0], u->ev[1]));
  UN_HIP(hipEventElapsedTime(&b, u->ev[1], u->ev[2]));
  u->fwd_ms = f;
  u->bwd_ms = b;
  if (loss) UN_HIP(hipMemcpy(loss, u->loss_dev, sizeof(double), hipMemcpyDeviceToHost));
  if (grad_host)
    UN_HIP(hipMemcpy(grad_host, u->grads, u->nparam * sizeof(float), hipMemcpyDeviceToHost));
  return XT_OK;
}

extern "C" int xt_unet_adam_step(xt_unet *u, float lr, float b1, float b2, float eps) {
  if (!u || !u->train) return xt_report_error(XT_E_ARG, "network has no training buffers");
  u->adam_t++;
  const float bc1 = 1.f - std::pow(b1, (float)u->adam_t), bc2 = 1.f - std::pow(b2, (float)u->adam_t);
  hipLaunchKernelGGL(k_adam, dim3(grid1(u->nparam)), dim3(256), 0, u->st, u->params, u->grads,
                     u->adam_m, u->adam_v, (size_t)u->nparam, lr, b1, b2, eps, bc1, bc2);
  UN_HIP(hipGetLastError());
  u->wdirty = true;
  UN_HIP(hipStreamSynchronize(u->st));
  return XT_OK;
}

extern "C" int xt_unet_train_step(xt_unet *u, const float *in, const float *tgt, float lr,
                                  double *loss) {
  UN_TRY(xt_unet_loss_grad(u, in, tgt, loss, nullptr));
  return xt_unet_adam_step(u, lr, 0.9f, 0.999f, 1e-8f);
}

static int stage_in(xt_unet *u, const float *a, const float *b) {
  if (!u->stage) UN_HIP(hipMalloc((void **)&u->stage, 2 * u->V[0] * sizeof(float)));
  UN_HIP(hipMemcpy(u->stage, a, u->V[0] * sizeof(float), hipMemcpyHostToDevice));
  if (b) UN_HIP(hipMemcpy(u->stage + u->V[0], b, u->V[0] * sizeof(float), hipMemcpyHostToDevice));
  return XT_OK;
}

extern "C" int xt_unet_forward_host(xt_unet *u, const float *in, float *out) {
  if (!u || !in || !out) return xt_report_error(XT_E_ARG, "null argument");
  UN_TRY(stage_in(u, in, nullptr));
  UN_TRY(xt_unet_forward(u, u->stage, u->stage + u->V[0]));
  UN_HIP(hipMemcpy(out, u->stage + u->V[0], u->V[0] * sizeof(float), hipMemcpyDeviceToHost));
  return XT_OK;
}

extern "C" int xt_unet_loss_grad_host(xt_unet *u, const float *in, const float *tgt, double *loss,
                                      float *grad_host) {
  if (!u || !in || !tgt) return xt_report_error(XT_E_ARG, "null argument");
  UN_TRY(stage_in(u, in, tgt));
  return xt_unet_loss_grad(u, u->stage, u->stage + u->V[0], loss, grad_host);
}

extern "C" int xt_unet_train_step_host(xt_unet *u, const float *in, const float *tgt, float lr,
                                       double *loss) {
  if (!u || !in || !tgt) return xt_report_error(XT_E_ARG, "null argument");
  UN_TRY(stage_in(u, in, tgt));
  return xt_unet_train_step(u, u->stage, u->stage + u->V[0], lr, loss);
}

extern "C" int xt_unet_last_ms(const xt_unet *u, double *fwd_ms, double *bwd_ms) {
  if (!u) return xt_report_error(XT_E_ARG, "null net");
  if (fwd_ms) *fwd_ms = u->fwd_ms;
  if (bwd_ms) *bwd_ms = u->bwd_ms;
  return XT_OK;
}
