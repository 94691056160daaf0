// Learned potential predictor: a 3-level periodic U-Net with BF16 MFMA inference and
// training kernels (C ABI in include/salmon_unet.h).
//
// Tensors are channels-last (point-major, channel fastest), p = ix + nx*(iy + ny*iz).
// Activations and MFMA operands are BF16 (round to nearest even), sums FP32.
//
//   x0 (16 ch: 4 inputs + zero pad)            level 0 (n)
//   e1a = relu(conv(x0)) 16, e1b = relu(conv(e1a)) 16
//   p1 = avgpool(e1b)                          level 1 (n/2)
//   e2a = relu(conv(p1)) 32, e2b = relu(conv(e2a)) 32
//   p2 = avgpool(e2b)                          level 2 (n/4)
//   e3a = relu(conv(p2)) 64, e3b = relu(conv(e3a)) 64
//   d2a = relu(conv([up(e3b), e2b])) 32, d2b = relu(conv(d2a)) 32      level 1
//   d1a = relu(conv([up(d2b), e1b])) 16, d1b = relu(conv(d1a)) 16      level 0
//   out = head(d1b) (1x1x1, FP32)
// conv = 3x3x3 periodic, weights [27][co][ci]; `up` = nearest upsampling, read on the fly.
//
// Kernels:
//   k_conv<NT,SK,CI>  implicit GEMM on gfx950's double-K v_mfma_f32_16x16x32_bf16: M = 16
//                  points per wave, N = NT x 16 output channels, K = 32 of the flattened
//                  (tap, input channel) index (two taps per instruction at 16 channels);
//                  also the data gradient (flipped, transposed weights; FP32 output, or masked by
//                  the activation)
//   k_wg_pack, k_wgrad, k_wg_reduce  weight and bias gradient as MFMA over points (M = co, N = ci, K = 32
//                  points of channel-major copies), FP32 partials reduced in fixed order
//   small kernels  pooling, gradient routing (down-sum, pool-back), head, MSE, Adam
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "salmon_hip.h"
#include "salmon_unet.h"

void salmon_hip_internal_error(const char *msg);  // salmon_hip.hip: sets salmon_hip_last_error()

namespace {

typedef unsigned short bf16_t;
typedef short s8v __attribute__((ext_vector_type(8)));
typedef __bf16 b8v __attribute__((ext_vector_type(8)));
typedef float f4v __attribute__((ext_vector_type(4)));

// v_mfma_f32_16x16x32_bf16 (gfx950): lane L holds A[L%16][8(L/16) + e] and
// B[8(L/16) + e][L%16], e = 0..7; D[4(L/16) + r][L%16] lands in register r.
__device__ __forceinline__ f4v mfma32(s8v a, s8v b, f4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8v, a), __builtin_bit_cast(b8v, b), c, 0, 0, 0);
}

int ufail(int code, const char *fmt, ...);

#define UHIP(x)                                                                               \
  do {                                                                                        \
    hipError_t e_ = (x);                                                                      \
    if (e_ != hipSuccess) return ufail(SALMON_HIP_EHIP, "%s: %s", #x, hipGetErrorString(e_)); \
  } while (0)
#define ULAUNCH(name)                                                                                   \
  do {                                                                                                  \
    hipError_t e_ = hipGetLastError();                                                                  \
    if (e_ != hipSuccess) return ufail(SALMON_HIP_EHIP, "launch %s: %s", name, hipGetErrorString(e_)); \
  } while (0)

__device__ __forceinline__ bf16_t f2bf(float f) {
  unsigned u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (bf16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(bf16_t h) { return __uint_as_float((unsigned)h << 16); }

// ---------------------------------------------------------------------------
// 3x3x3 periodic convolution as implicit GEMM.  Wave w of block b owns points
// p0 = 16 (4b + w) .. p0 + 15; A row = point, B col = output channel, K = the
// flattened index f = tap * ci + input channel.  One MFMA takes 32 consecutive f:
// lane group q = L/16 supplies f0 + 8q .. f0 + 8q + 7, which lie in one tap and one
// 16-channel chunk (ci is a multiple of 16), i.e. one 16-byte load of activations at
// the tap's neighbour and one of weights.  The input is [up(src1), src2] (channel
// concatenation, src1 at half resolution when up1).
// ---------------------------------------------------------------------------
constexpr size_t kConvZero = 128 * 128 + 64;  // bf16 zeros read by k_conv (co x ci up to 128 x 128)

struct ConvArgs {
  const bf16_t *src1, *src2;
  int c1, c2, up1;
  const bf16_t *w;      // [27][co][c1 + c2]
  const float *bias;    // [co] or null
  const bf16_t *mask;   // [npts][co]: results where it is not above 0 are 0 (the gradient of relu), or null
  bf16_t *out_bf;       // [npts][co] (bias, optional relu, mask), or
  float *out_f;         // [npts][co] raw
  int co, relu;
  int nx, ny, nz, npts;
  const bf16_t *zero;   // zero-filled, at least co * (c1 + c2) + 8 elements
};

// SK = false: each wave takes its own 16 points and the whole K; SK = true (coarse levels, few
// points): the four waves of a block share 16 points and take every fourth K step each, and wave
// 0 adds the four partial sums in a fixed order (deterministic).
//
// CI = input channels / 16.  Bound by the latency of the operand loads (a wave has 2 (1 + NT) KB of
// operands per K step and 14 to 81 steps): U steps' loads are issued together, the next group's while the
// MFMAs of a group run, and the channel count is a constant so that a step's addresses cost no division.
// With one step ahead and runtime divisions a 16 -> 16 layer took 12.7 us at 32^3, now 6.2.
// blockIdx.y takes NT output tiles each: with SK one per block, as a coarse level's points alone leave most
// CUs idle (64 -> 64 channels at 8^3 13.8 us with four tiles per wave, 6.5 us so).
template <int NT, bool SK, int CI>
__global__ __launch_bounds__(256) void k_conv(ConvArgs a) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int p0 = (SK ? blockIdx.x : blockIdx.x * 4 + wave) * 16;
  if (p0 >= a.npts) return;
  const int row = lane & 15, kq = lane >> 4;
  const int ct = blockIdx.y * NT * 16;  // first output channel of this block
  const int p = p0 + row;
  const bool pv = p < a.npts;
  const int pp = pv ? p : 0;
  const int nx = a.nx, ny = a.ny, nz = a.nz;
  const int x = pp % nx, y = (pp / nx) % ny, z = pp / (nx * ny);
  constexpr int ci = 16 * CI, K = 27 * ci;
  f4v acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f4v{0.f, 0.f, 0.f, 0.f};
  // the operands of K step f0 (32 wide: lane group kq takes f0 + 8 kq .. + 7)
  // (branch-free: what lies outside the point range or past K is read from a zero buffer, so
  // every lane issues the same loads and each wait can sit at the MFMA that uses the data)
  auto load = [&](int f0, s8v &av, s8v (&bv)[NT]) __attribute__((always_inline)) {
    const unsigned f = f0 + 8 * kq;
    const bool fv = f < K;
    const unsigned fc = fv ? f : 0;
    const int tap = fc / ci, c = fc - tap * ci;
    const int dz = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dx = tap % 3 - 1;
    int xn = x + dx, yn = y + dy, zn = z + dz;
    xn += xn < 0 ? nx : 0;
    xn -= xn >= nx ? nx : 0;
    yn += yn < 0 ? ny : 0;
    yn -= yn >= ny ? ny : 0;
    zn += zn < 0 ? nz : 0;
    zn -= zn >= nz ? nz : 0;
    const int pn = xn + nx * (yn + ny * zn);
    const int ph = a.up1 ? (xn >> 1) + (nx >> 1) * ((yn >> 1) + (ny >> 1) * (zn >> 1)) : pn;
    const bf16_t *src = c < a.c1 ? a.src1 + (size_t)ph * a.c1 + c : a.src2 + (size_t)pn * a.c2 + (c - a.c1);
    av = *(const s8v *)((fv && pv) ? src : a.zero);
    const bf16_t *wt = fv ? a.w + (size_t)(tap * a.co) * ci + c : a.zero;
#pragma unroll
    for (int t = 0; t < NT; ++t) bv[t] = *(const s8v *)(wt + (ct + t * 16 + row) * ci);
  };
  // this wave's K steps fs, fs + kst, ... in two sets of U operands (steps past the end multiply zeros
  // and are left out); the accumulation order is that of the steps
  constexpr int kst = SK ? 4 * 32 : 32;
  constexpr int U = NT == 1 ? 7 : NT == 2 ? 5 : NT == 3 ? 4 : NT == 4 ? 3 : 2;
  const int fs = SK ? 32 * wave : 0;
  s8v av[2][U], bv[2][U][NT];
  auto load_group = [&](int f0, s8v (&A)[U], s8v (&B)[U][NT]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u) load(f0 + kst * u, A[u], B[u]);
  };
  auto mfma_group = [&](int f0, s8v (&A)[U], s8v (&B)[U][NT]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (f0 + kst * u < K)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = mfma32(A[u], B[u][t], acc[t]);
  };
  load_group(fs, av[0], bv[0]);
  for (int f0 = fs; f0 < K; f0 += 2 * U * kst) {
    if (f0 + U * kst < K) load_group(f0 + U * kst, av[1], bv[1]);
    mfma_group(f0, av[0], bv[0]);
    if (f0 + U * kst >= K) break;
    if (f0 + 2 * U * kst < K) load_group(f0 + 2 * U * kst, av[0], bv[0]);
    mfma_group(f0 + U * kst, av[1], bv[1]);
  }
  if constexpr (SK) {
    __shared__ f4v red[3][NT][64];
    if (wave > 0)
#pragma unroll
      for (int t = 0; t < NT; ++t) red[wave - 1][t][lane] = acc[t];
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = ((acc[t] + red[0][t][lane]) + red[1][t][lane]) + red[2][t][lane];
  }
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int pr = p0 + 4 * kq + r;
      const int ch = ct + t * 16 + row;
      if (pr >= a.npts) continue;
      float v = acc[t][r];
      if (a.out_bf) {
        if (a.bias) v += a.bias[ch];
        if (a.relu) v = fmaxf(v, 0.f);
        if (a.mask && !(bf2f(a.mask[(size_t)pr * a.co + ch]) > 0.f)) v = 0.f;
        a.out_bf[(size_t)pr * a.co + ch] = f2bf(v);
      } else {
        a.out_f[(size_t)pr * a.co + ch] = v;
      }
    }
}

// ---------------------------------------------------------------------------
// Weight and bias gradient of a convolution: dW[tap][co][ci] = sum_p dy[p][co] x[p + d(tap)][ci],
// db[co] = sum_p dy[p][co].  The MFMAs' K runs over points, so an operand is 8 consecutive points of
// one channel per lane: k_wg_pack first lays both tensors out channel-major, the input three times,
// shifted by -1, 0 and 1 along x with its periodic neighbour.  A wave then takes one (dz, dy) of the
// kernel, 16 input channels, one or two tiles of 16 output channels and 1024 points: an 8-point block is
// one 16-byte load where rows are whole blocks (8 / G loads of G points where only G divides the row
// length: a group of G never spans two rows, so its neighbour rows are contiguous too), and each block of
// dy serves the three dx taps.  Points are summed in the order of their index, 32 per MFMA, the 1024-point
// shares in ascending order (k_wg_reduce).
//
// A wave per (tap, co tile, ci tile) gathering single 2-byte elements, three divisions each, took 91 us
// per layer on average at 32^3 where the three kernels here take 20 (4 + 11 + 5) a layer at a time, bound
// by the latency of the loads (288 waves at the finest level's 16 x 16 channels), not by the matrix
// cores; all ten layers of a sample in one launch each take 74 us instead of 198 (11 + 54 + 10).
// ---------------------------------------------------------------------------
constexpr int kWgChunk = 1024;  // points per partial sum

struct WgArgs {
  const bf16_t *dy;            // [npts][co]
  int co;
  const bf16_t *src1, *src2;   // input [up(src1), src2], channels-last
  int c1, c2, up1;
  bf16_t *xt;                  // [3][ci][npad]
  bf16_t *gt;                  // [co][npad]
  float *part;                 // [chunks][27][co][ci]
  float *grad;                 // [27 co ci weights][co biases]
  int nx, ny, nz, npts, npad;  // npad: npts rounded up to whole 32-point steps (zeros past npts)
};

// Several layers in one launch: layer i owns the blocks [off[i], off[i + 1]).
constexpr int kWgLayers = 10;
struct WgAll {
  WgArgs l[kWgLayers];
  unsigned off[kWgLayers + 1];
  int n;
};

__device__ __forceinline__ int wg_layer(const WgAll &A, unsigned b) {
  int i = 0;
  while (i + 1 < A.n && b >= A.off[i + 1]) ++i;
  return i;
}

// one thread per (point, 8 channels): the input's threads, then dy's
__global__ __launch_bounds__(256) void k_wg_pack(WgAll A) {
  const int li = wg_layer(A, blockIdx.x);
  const WgArgs &a = A.l[li];
  const int ci = a.c1 + a.c2;
  const size_t nxi = (size_t)a.npad * (ci / 8);
  size_t i = (size_t)(blockIdx.x - A.off[li]) * 256 + threadIdx.x;
  const s8v zero = {0, 0, 0, 0, 0, 0, 0, 0};
  if (i < nxi) {
    const int p = i % a.npad, c = 8 * (int)(i / a.npad);
    const size_t plane = (size_t)ci * a.npad;
    const int x = p % a.nx, r = p / a.nx;
    const int y = r % a.ny, z = r / a.ny;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      int xn = x + d - 1;
      xn += xn < 0 ? a.nx : 0;
      xn -= xn >= a.nx ? a.nx : 0;
      s8v v = zero;
      if (p < a.npts) {
        if (c < a.c1) {
          const size_t q = a.up1 ? (size_t)(xn >> 1) + (size_t)(a.nx >> 1) * ((size_t)(y >> 1) + (size_t)(a.ny >> 1) * (z >> 1))
                                 : (size_t)xn + (size_t)a.nx * r;
          v = *(const s8v *)(a.src1 + q * a.c1 + c);
        } else {
          v = *(const s8v *)(a.src2 + ((size_t)xn + (size_t)a.nx * r) * a.c2 + (c - a.c1));
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) a.xt[d * plane + (size_t)(c + e) * a.npad + p] = (bf16_t)v[e];
    }
    return;
  }
  i -= nxi;
  if (i >= (size_t)a.npad * (a.co / 8)) return;
  const int p = i % a.npad, c = 8 * (int)(i / a.npad);
  const s8v v = p < a.npts ? *(const s8v *)(a.dy + (size_t)p * a.co + c) : zero;
#pragma unroll
  for (int e = 0; e < 8; ++e) a.gt[(size_t)(c + e) * a.npad + p] = (bf16_t)v[e];
}

template <int G> struct WgGroup;
template <> struct WgGroup<8> { typedef s8v T; };
template <> struct WgGroup<4> { typedef short T __attribute__((ext_vector_type(4))); };
template <> struct WgGroup<2> { typedef short T __attribute__((ext_vector_type(2))); };
template <> struct WgGroup<1> { typedef short T; };

// NCO: output tiles per wave; G: points per load of the input (a divisor of nx)
template <int NCO, int G>
__global__ __launch_bounds__(64) void k_wgrad(WgAll A) {
  const int li = wg_layer(A, blockIdx.x);
  const WgArgs &a = A.l[li];
  const int lane = threadIdx.x;
  const int row = lane & 15, kq = lane >> 4;
  const int ci = a.c1 + a.c2;
  const int nci = ci / 16, nct = a.co / 16 / NCO;
  int t = blockIdx.x - A.off[li];
  const int cit = t % nci;
  t /= nci;
  const int cot = NCO * (t % nct);
  t /= nct;
  const int g = t % 9, chunk = t / 9;
  const int dz = g / 3 - 1, dyy = g % 3 - 1;
  const int pbeg = chunk * kWgChunk, pend = min(pbeg + kWgChunk, a.npts);
  f4v acc[3][NCO];
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int k = 0; k < NCO; ++k) acc[d][k] = f4v{0.f, 0.f, 0.f, 0.f};
  const size_t plane = (size_t)ci * a.npad;
  const bf16_t *xr = a.xt + (size_t)(cit * 16 + row) * a.npad;
  const bf16_t *gr = a.gt + (size_t)(cot * 16 + row) * a.npad;
  // p / nx by a reciprocal multiply with one correction step
  const float rnx = 1.f / (float)a.nx, rny = 1.f / (float)a.ny;
  auto divide = [](int p, int n, float rn) __attribute__((always_inline)) {
    int q = (int)((float)p * rn);
    q += (q + 1) * n <= p ? 1 : 0;
    q -= q * n > p ? 1 : 0;
    return q;
  };
  typedef typename WgGroup<G>::T T;
  auto load = [&](int pb, s8v (&av)[NCO], s8v (&bv)[3]) __attribute__((always_inline)) {
    const int p0 = min(pb + 8 * kq, a.npad - 8);  // the lane's 8 points (dy is zero past npts)
#pragma unroll
    for (int k = 0; k < NCO; ++k) av[k] = *(const s8v *)(gr + (size_t)(16 * k) * a.npad + p0);
#pragma unroll
    for (int h = 0; h < 8 / G; ++h) {
      const int p = min(p0 + G * h, a.npts - G);
      const int r = divide(p, a.nx, rnx);
      const int x = p - r * a.nx;
      const int z = divide(r, a.ny, rny);
      int yn = r - z * a.ny + dyy, zn = z + dz;
      yn += yn < 0 ? a.ny : 0;
      yn -= yn >= a.ny ? a.ny : 0;
      zn += zn < 0 ? a.nz : 0;
      zn -= zn >= a.nz ? a.nz : 0;
      const bf16_t *xp = xr + (size_t)(zn * a.ny + yn) * a.nx + x;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        if constexpr (G == 8) {
          bv[d] = *(const s8v *)(xp + d * plane);
        } else if constexpr (G == 1) {
          bv[d][h] = (short)xp[d * plane];
        } else {
          const T v = *(const T *)(xp + d * plane);
#pragma unroll
          for (int e = 0; e < G; ++e) bv[d][G * h + e] = v[e];
        }
      }
    }
  };
  // two sets of U steps: the next set's loads are in flight while a set's MFMAs run
  constexpr int U = NCO == 1 ? 6 : 5;
  s8v av[2][U][NCO], bv[2][U][3];
  auto load_group = [&](int pb, s8v (&A)[U][NCO], s8v (&B)[U][3]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u) load(pb + 32 * u, A[u], B[u]);
  };
  auto mfma_group = [&](int pb, s8v (&A)[U][NCO], s8v (&B)[U][3]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (pb + 32 * u < pend)
#pragma unroll
        for (int k = 0; k < NCO; ++k)
#pragma unroll
          for (int d = 0; d < 3; ++d) acc[d][k] = mfma32(A[u][k], B[u][d], acc[d][k]);
  };
  load_group(pbeg, av[0], bv[0]);
  for (int pb = pbeg; pb < pend; pb += 64 * U) {
    if (pb + 32 * U < pend) load_group(pb + 32 * U, av[1], bv[1]);
    mfma_group(pb, av[0], bv[0]);
    if (pb + 32 * U >= pend) break;
    if (pb + 64 * U < pend) load_group(pb + 64 * U, av[0], bv[0]);
    mfma_group(pb + 32 * U, av[1], bv[1]);
  }
  float *part = a.part + (size_t)chunk * 27 * a.co * ci;
#pragma unroll
  for (int k = 0; k < NCO; ++k)
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        part[((size_t)(3 * g + d) * a.co + (cot + k) * 16 + 4 * kq + e) * ci + cit * 16 + row] = acc[d][k][e];
}

// grad[i] += sum_k part[k][i], k ascending, 8 loads in flight (a layer's first nwb blocks), and the biases:
// grad[nw + c] += sum_p dy[p][c], one block per channel, fixed-order tree
__global__ __launch_bounds__(256) void k_wg_reduce(WgAll A) {
  __shared__ float sh[256];
  const int li = wg_layer(A, blockIdx.x);
  const WgArgs &a = A.l[li];
  const unsigned bx = blockIdx.x - A.off[li];
  const int nk = (a.npts + kWgChunk - 1) / kWgChunk;
  const size_t nw = (size_t)27 * a.co * (a.c1 + a.c2);
  const unsigned nwb = (unsigned)((nw + 255) / 256);
  if (bx < nwb) {
    const size_t i = (size_t)bx * 256 + threadIdx.x;
    if (i >= nw) return;
    float s = 0.f;
    for (int k = 0; k < nk; k += 8) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = a.part[(size_t)min(k + u, nk - 1) * nw + i];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (k + u < nk) s += v[u];
    }
    a.grad[i] += s;
    return;
  }
  const int c = bx - nwb;
  const bf16_t *g = a.gt + (size_t)c * a.npad;
  float s = 0.f;
  for (int p0 = threadIdx.x; p0 < a.npts; p0 += 256 * 16) {
    bf16_t v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) v[u] = g[min(p0 + 256 * u, a.npts - 1)];
#pragma unroll
    for (int u = 0; u < 16; ++u)
      if (p0 + 256 * u < a.npts) s += bf2f(v[u]);
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) sh[threadIdx.x] += sh[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) a.grad[nw + c] += sh[0];
}

// 2x2x2 average pool: out (hx, hy, hz) = mean of its 8 children
__global__ __launch_bounds__(256) void k_pool(const bf16_t *in, bf16_t *out, int hx, int hy, int hz, int C) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  const size_t n = (size_t)hx * hy * hz * C;
  if (i >= n) return;
  const int c = i % C;
  const size_t q = i / C;
  const int x = q % hx, y = (q / hx) % hy, z = q / ((size_t)hx * hy);
  const int nx = 2 * hx, ny = 2 * hy;
  float s = 0.f;
  for (int k = 0; k < 8; ++k) {
    const int xx = 2 * x + (k & 1), yy = 2 * y + ((k >> 1) & 1), zz = 2 * z + (k >> 2);
    s += bf2f(in[((size_t)xx + (size_t)nx * ((size_t)yy + (size_t)ny * zz)) * C + c]);
  }
  out[i] = f2bf(s * 0.125f);
}

// out[q][c] = bf16((sum of the 8 children of q of gin[.][c]) * (act[q][c] > 0)) (gradient of nearest upsampling)
__global__ __launch_bounds__(256) void k_downsum(const float *gin, int Cs, int C, const bf16_t *act, bf16_t *out, int hx,
                                                 int hy, int hz) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  const size_t n = (size_t)hx * hy * hz * C;
  if (i >= n) return;
  const int c = i % C;
  const size_t q = i / C;
  const int x = q % hx, y = (q / hx) % hy, z = q / ((size_t)hx * hy);
  const int nx = 2 * hx, ny = 2 * hy;
  float s = 0.f;
  for (int k = 0; k < 8; ++k) {
    const int xx = 2 * x + (k & 1), yy = 2 * y + ((k >> 1) & 1), zz = 2 * z + (k >> 2);
    s += gin[((size_t)xx + (size_t)nx * ((size_t)yy + (size_t)ny * zz)) * Cs + c];
  }
  out[i] = f2bf(bf2f(act[i]) > 0.f ? s : 0.f);
}

// out[p][c] = bf16((gp[parent(p)][c] / 8 + gskip[p][off + c]) * (act[p][c] > 0))
__global__ __launch_bounds__(256) void k_poolback(const float *gp, const float *gskip, int Cs, int off, int C,
                                                  const bf16_t *act, int nx, int ny, int nz, bf16_t *out) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  const size_t n = (size_t)nx * ny * nz * C;
  if (i >= n) return;
  const int c = i % C;
  const size_t p = i / C;
  const int x = p % nx, y = (p / nx) % ny, z = p / ((size_t)nx * ny);
  const size_t q = (size_t)(x >> 1) + (size_t)(nx >> 1) * ((size_t)(y >> 1) + (size_t)(ny >> 1) * (z >> 1));
  float v = gp[q * C + c] * 0.125f;
  if (gskip) v += gskip[p * Cs + off + c];
  if (!(bf2f(act[i]) > 0.f)) v = 0.f;
  out[i] = f2bf(v);
}

__global__ __launch_bounds__(256) void k_pack_input(const float *in, size_t npts, bf16_t *x0) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= npts * 16) return;
  const size_t p = i / 16;
  const int c = i % 16;
  x0[i] = c < 4 ? f2bf(in[p * 4 + c]) : (bf16_t)0;
}

// out[p] = sum_c x[p][c] wh[c] + bh
__global__ __launch_bounds__(256) void k_head(const bf16_t *x, const float *wh, size_t npts, float *out) {
  const size_t p = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= npts) return;
  float s = 0.f;
  for (int c = 0; c < 16; ++c) s += bf2f(x[p * 16 + c]) * wh[c];
  out[p] = s + wh[16];
}

// dout[p] = 2 (out - t) / n; part[block] = sum (out - t)^2 over the block
__global__ __launch_bounds__(256) void k_mse(const float *out, const float *t, size_t n, float *dout, float *part) {
  __shared__ float sh[256];
  const size_t p = (size_t)blockIdx.x * 256 + threadIdx.x;
  float e2 = 0.f;
  if (p < n) {
    const float d = out[p] - t[p];
    dout[p] = 2.f * d / (float)n;
    e2 = d * d;
  }
  sh[threadIdx.x] = e2;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) sh[threadIdx.x] += sh[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

__global__ __launch_bounds__(256) void k_loss(const float *part, int nb, size_t n, float *loss) {
  __shared__ float sh[256];
  float s = 0.f;
  for (int k = threadIdx.x; k < nb; k += 256) s += part[k];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) sh[threadIdx.x] += sh[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) *loss = sh[0] / (float)n;
}

// head gradients: block b < 4: grad[c] += sum_p dout[p] x[p][c] for its four channels; block 4: grad[16]
// += sum dout.  A thread takes every 256th point, one 8-byte load for its channels, 8 points in flight;
// fixed-order tree.  (One block and one 2-byte load per channel: 42 us at 32^3, 14 us here.)
__global__ __launch_bounds__(256) void k_head_grad(const float *dout, const bf16_t *x, size_t npts, float *grad) {
  __shared__ float sh[4][256];
  typedef short s4v __attribute__((ext_vector_type(4)));
  const bool ones = blockIdx.x == 4;
  const int c0 = ones ? 0 : 4 * blockIdx.x;
  float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (size_t p = threadIdx.x; p < npts; p += 256) {
    const float d = dout[p];
    const s4v v = *(const s4v *)(x + p * 16 + c0);
#pragma unroll
    for (int c = 0; c < 4; ++c) s[c] += d * (ones ? 1.f : bf2f((bf16_t)v[c]));
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) sh[c][threadIdx.x] = s[c];
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k)
#pragma unroll
      for (int c = 0; c < 4; ++c) sh[c][threadIdx.x] += sh[c][threadIdx.x + k];
    __syncthreads();
  }
  if (ones && threadIdx.x == 0) grad[16] += sh[0][0];
  if (!ones && threadIdx.x < 4) grad[c0 + threadIdx.x] += sh[threadIdx.x][0];
}

// g[p][c] = bf16(dout[p] wh[c] (act[p][c] > 0))
__global__ __launch_bounds__(256) void k_head_back(const float *dout, const float *wh, const bf16_t *act, size_t npts,
                                                   bf16_t *g) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= npts * 16) return;
  const size_t p = i / 16;
  const int c = i % 16;
  g[i] = f2bf(bf2f(act[i]) > 0.f ? dout[p] * wh[c] : 0.f);
}

__global__ __launch_bounds__(256) void k_adam(size_t n, float *w, float *g, float *m, float *v, float lr, float c1,
                                              float c2, float inv_ns) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i] * inv_ns;
  const float mi = 0.9f * m[i] + 0.1f * gi;
  const float vi = 0.999f * v[i] + 0.001f * gi * gi;
  m[i] = mi;
  v[i] = vi;
  w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + 1e-8f);
  g[i] = 0.f;
}

// wt[tap][co][ci] = bf16(w), wb[26 - tap][ci][co] = bf16(w) (data-gradient weights), all layers: layer i owns
// the blocks [off[i], off[i + 1])
struct PackArgs {
  const float *w[kWgLayers];
  bf16_t *wt[kWgLayers], *wb[kWgLayers];
  int co[kWgLayers], ci[kWgLayers];
  unsigned off[kWgLayers + 1];
};

__global__ __launch_bounds__(256) void k_pack_w(PackArgs A) {
  int li = 0;
  while (li + 1 < kWgLayers && blockIdx.x >= A.off[li + 1]) ++li;
  const int co = A.co[li], ci = A.ci[li];
  const size_t i = (size_t)(blockIdx.x - A.off[li]) * 256 + threadIdx.x;
  if (i >= (size_t)27 * co * ci) return;
  const int c = i % ci;
  const int o = (i / ci) % co;
  const int tap = i / ((size_t)co * ci);
  const bf16_t h = f2bf(A.w[li][i]);
  A.wt[li][i] = h;
  A.wb[li][((size_t)(26 - tap) * ci + c) * co + o] = h;
}

// ---------------------------------------------------------------------------
// Predictor glue on FP64 potentials V_local(ix,iy,iz), history v0 = V(t), v1 = V(t-dt), ...
// ---------------------------------------------------------------------------
// in[p] = ((v0 - v1)/sd, (v1 - v2)/sd, (v2 - v3)/sd, (v0 - vpsl)/sa)
__global__ __launch_bounds__(256) void k_features(const double *v0, const double *v1, const double *v2,
                                                  const double *v3, const double *vpsl, double sd, double sa,
                                                  size_t n, float *in) {
  const size_t p = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= n) return;
  const double a = v0[p], b = v1[p], c = v2[p], d = v3[p];
  in[4 * p + 0] = (float)((a - b) / sd);
  in[4 * p + 1] = (float)((b - c) / sd);
  in[4 * p + 2] = (float)((c - d) / sd);
  in[4 * p + 3] = (float)((a - vpsl[p]) / sa);
}

// vpred = v0 + (v0 - v1)/2 + so * nn   (linear extrapolation to t + dt/2 plus the learned correction)
__global__ __launch_bounds__(256) void k_predict(const double *v0, const double *v1, const float *nn, double so,
                                                 size_t n, double *vpred) {
  const size_t p = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= n) return;
  const double a = v0[p];
  vpred[p] = a + 0.5 * (a - v1[p]) + so * (double)nn[p];
}

// t = (vmid - v0 - (v0 - v1)/2) / so
__global__ __launch_bounds__(256) void k_target(const double *vmid, const double *v0, const double *v1, double so,
                                                size_t n, float *t) {
  const size_t p = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= n) return;
  const double a = v0[p];
  t[p] = (float)((vmid[p] - a - 0.5 * (a - v1[p])) / so);
}

// part[block] = max_p |vpred - (v0 + vnew)/2| over the block; out = max over blocks
__global__ __launch_bounds__(256) void k_resid_part(const double *vpred, const double *v0, const double *vnew, size_t n,
                                                    double *part) {
  __shared__ double sh[256];
  double m = 0.0;
  for (size_t p = (size_t)blockIdx.x * 256 + threadIdx.x; p < n; p += (size_t)gridDim.x * 256)
    m = fmax(m, fabs(vpred[p] - 0.5 * (v0[p] + vnew[p])));
  sh[threadIdx.x] = m;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) sh[threadIdx.x] = fmax(sh[threadIdx.x], sh[threadIdx.x + k]);
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

__global__ __launch_bounds__(256) void k_resid_final(const double *part, int nb, double *out) {
  __shared__ double sh[256];
  double m = 0.0;
  for (int k = threadIdx.x; k < nb; k += 256) m = fmax(m, part[k]);
  sh[threadIdx.x] = m;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) sh[threadIdx.x] = fmax(sh[threadIdx.x], sh[threadIdx.x + k]);
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = sh[0];
}

// The gate of a step propagated with a predicted potential, decided on the device: flag =
// (resid <= tol); stats[0] counts accepted, stats[1] attempted steps; log[stats[1]] = resid while
// the log has room.
__global__ void k_gate(const double *resid, double tol, int *flag, int *stats, double *log, int log_cap) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  const double r = *resid;
  const int ok = r <= tol ? 1 : 0;
  const int n = stats[1];
  if (log && n < log_cap) log[n] = r;
  *flag = ok;
  stats[0] += ok;
  stats[1] = n + 1;
}

int ufail(int code, const char *fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  salmon_hip_internal_error(buf);
  return code;
}

unsigned blocks(size_t n) { return (unsigned)((n + 255) / 256); }

struct Layer {
  int co, c1, c2, up1, level;  // input [up(src1) (c1), src2 (c2)] at `level`
  size_t woff, boff;           // offsets in the flat parameter array
  size_t xt_off, gt_off, part_off;  // its part of the weight gradients' work
  bf16_t *wt = nullptr, *wb = nullptr;
};

}  // namespace

struct salmon_unet {
  int n[3][3];   // grid extents per level
  size_t np[3];  // points per level
  hipStream_t stream = nullptr;
  std::vector<Layer> L;
  size_t nparam = 0, head_off = 0;
  float *d_w = nullptr, *d_g = nullptr, *d_m = nullptr, *d_v = nullptr;
  int adam_t = 0;
  bool packed = false;
  // activations (bf16): x0, e1a, e1b, p1, e2a, e2b, p2, e3a, e3b, d2a, d2b, d1a, d1b
  bf16_t *x0 = nullptr, *act[12] = {};
  bf16_t *d_zero = nullptr;  // kConvZero zeros: the operands of k_conv outside the grid or past K
  // backward work
  float *d_out = nullptr, *d_dout = nullptr, *d_part = nullptr;
  // the weight gradients run last: their operands and partial sums lie where the data gradients (d_fx with
  // d_xt) and, once packed, the layers' gradients (g with d_wpart) lay
  float *d_fx = nullptr, *d_wpart = nullptr;
  bf16_t *g[10] = {};        // pre-activation gradient of each layer
  bf16_t *d_xt = nullptr, *d_gt = nullptr;  // channel-major operands of the weight gradient
  size_t fx_n = 0;
  double *d_rpart = nullptr;  // residual partial maxima
  std::vector<void *> allocs;
};

namespace {

enum { E1A = 0, E1B, P1, E2A, E2B, P2, E3A, E3B, D2A, D2B, D1A, D1B };

template <typename T>
int ualloc(salmon_unet *u, T **p, size_t n) {
  *p = nullptr;
  if (hipMalloc((void **)p, sizeof(T) * std::max<size_t>(n, 1)) != hipSuccess)
    return ufail(SALMON_HIP_ENOMEM, "hipMalloc(%zu bytes) failed", sizeof(T) * n);
  u->allocs.push_back((void *)*p);
  return 0;
}

int launch_conv(salmon_unet *u, const bf16_t *s1, int c1, int up1, const bf16_t *s2, int c2, const bf16_t *w,
                const float *bias, int co, int relu, int level, bf16_t *out_bf, float *out_f,
                const bf16_t *mask = nullptr) {
  ConvArgs a;
  a.src1 = s1; a.src2 = s2; a.c1 = c1; a.c2 = c2; a.up1 = up1;
  a.w = w; a.bias = bias; a.mask = mask; a.out_bf = out_bf; a.out_f = out_f; a.co = co; a.relu = relu;
  a.nx = u->n[level][0]; a.ny = u->n[level][1]; a.nz = u->n[level][2];
  a.npts = (int)u->np[level];
  a.zero = u->d_zero;
  if ((size_t)co * (c1 + c2) + 8 > kConvZero)
    return ufail(SALMON_HIP_EUNSUPPORTED, "conv %d -> %d channels above the zero operand", c1 + c2, co);
  // fewer 64-point blocks than CUs: split K over the four waves of 16-point blocks, one tile of output
  // channels each
  const bool sk = (a.npts + 63) / 64 < 256;
  const unsigned nb = (unsigned)(sk ? (a.npts + 15) / 16 : (a.npts + 63) / 64);
#define CONV_LAUNCH(NTv, CIv)                                                                      \
  case 16 * NTv + CIv:                                                                             \
    if (sk) hipLaunchKernelGGL((k_conv<1, true, CIv>), dim3(nb, NTv), dim3(256), 0, u->stream, a); \
    else hipLaunchKernelGGL((k_conv<NTv, false, CIv>), dim3(nb), dim3(256), 0, u->stream, a);      \
    break
  // output and input tiles of the layers, forward and (transposed) backward
  switch (c1 % 16 == 0 && c2 % 16 == 0 && co % 16 == 0 ? co + (c1 + c2) / 16 : 0) {
    CONV_LAUNCH(1, 1);
    CONV_LAUNCH(1, 2);
    CONV_LAUNCH(1, 3);
    CONV_LAUNCH(2, 1);
    CONV_LAUNCH(2, 2);
    CONV_LAUNCH(2, 4);
    CONV_LAUNCH(2, 6);
    CONV_LAUNCH(3, 1);
    CONV_LAUNCH(4, 2);
    CONV_LAUNCH(4, 4);
    CONV_LAUNCH(6, 2);
    default: return ufail(SALMON_HIP_EUNSUPPORTED, "conv %d -> %d channels", c1 + c2, co);
  }
#undef CONV_LAUNCH
  ULAUNCH("k_conv");
  return 0;
}

const bf16_t *layer_src1(salmon_unet *u, int i) {
  static const int src[12] = {-1, E1A, -2, P1, E2A, -2, P2, E3A, E3B, D2A, D2B, D1A};
  return src[i] == -1 ? u->x0 : u->act[src[i]];
}
const bf16_t *layer_src2(salmon_unet *u, int i) {
  if (i == D2A) return u->act[E2B];
  if (i == D1A) return u->act[E1B];
  return nullptr;
}

int pack_weights(salmon_unet *u) {
  PackArgs A;
  A.off[0] = 0;
  for (int li = 0; li < kWgLayers; ++li) {
    const Layer &l = u->L[li];
    A.w[li] = u->d_w + l.woff;
    A.wt[li] = l.wt;
    A.wb[li] = l.wb;
    A.co[li] = l.co;
    A.ci[li] = l.c1 + l.c2;
    A.off[li + 1] = A.off[li] + blocks((size_t)27 * l.co * (l.c1 + l.c2));
  }
  hipLaunchKernelGGL(k_pack_w, dim3(A.off[kWgLayers]), dim3(256), 0, u->stream, A);
  ULAUNCH("k_pack_w");
  u->packed = true;
  return 0;
}

int forward(salmon_unet *u, const float *in, float *out) {
  if (!u->packed)
    if (int rc = pack_weights(u)) return rc;
  hipLaunchKernelGGL(k_pack_input, dim3(blocks(u->np[0] * 16)), dim3(256), 0, u->stream, in, u->np[0], u->x0);
  ULAUNCH("k_pack_input");
  int li = 0;
  for (int i = 0; i < 12; ++i) {
    if (i == P1 || i == P2) {
      const int lv = i == P1 ? 1 : 2;
      const int C = i == P1 ? 16 : 32;
      hipLaunchKernelGGL(k_pool, dim3(blocks(u->np[lv] * C)), dim3(256), 0, u->stream, u->act[i - 1], u->act[i],
                         u->n[lv][0], u->n[lv][1], u->n[lv][2], C);
      ULAUNCH("k_pool");
      continue;
    }
    Layer &l = u->L[li++];
    if (int rc = launch_conv(u, layer_src1(u, i), l.c1, l.up1, layer_src2(u, i), l.c2, l.wt, u->d_w + l.boff, l.co, 1,
                             l.level, u->act[i], nullptr))
      return rc;
  }
  hipLaunchKernelGGL(k_head, dim3(blocks(u->np[0])), dim3(256), 0, u->stream, u->act[D1B], u->d_w + u->head_off,
                     u->np[0], out);
  ULAUNCH("k_head");
  return 0;
}

size_t wg_pad(size_t npts) { return (npts + 31) / 32 * 32; }

// weight and bias gradient of conv layer li (act index i) from its pre-activation gradient
WgArgs wg_args(salmon_unet *u, int li, int i) {
  const Layer &l = u->L[li];
  WgArgs a;
  a.dy = u->g[li]; a.co = l.co;
  a.src1 = layer_src1(u, i); a.src2 = layer_src2(u, i); a.c1 = l.c1; a.c2 = l.c2; a.up1 = l.up1;
  a.xt = u->d_xt + l.xt_off; a.gt = u->d_gt + l.gt_off;
  a.part = u->d_wpart + l.part_off;
  a.grad = u->d_g + l.woff;  // the layer's weights and biases lie side by side
  a.nx = u->n[l.level][0]; a.ny = u->n[l.level][1]; a.nz = u->n[l.level][2];
  a.npts = (int)u->np[l.level];
  a.npad = (int)wg_pad(a.npts);
  return a;
}

void wg_add(WgAll &A, const WgArgs &a, size_t nblk) {
  if (A.n == 0) A.off[0] = 0;
  A.l[A.n] = a;
  A.off[A.n + 1] = A.off[A.n] + (unsigned)nblk;
  ++A.n;
}

// Weight and bias gradients of all layers once their pre-activation gradients stand: three launches (the
// main one split by the two forms below), where one layer alone leaves most of the chip idle.
int weight_grads(salmon_unet *u, const int *conv_act) {
  WgAll P, R, W[2][4];
  P.n = R.n = 0;
  for (auto &w : W)
    for (WgAll &x : w) x.n = 0;
  for (int li = 9; li >= 0; --li) {
    const WgArgs a = wg_args(u, li, conv_act[li]);
    const int ci = a.c1 + a.c2;
    const size_t nw = (size_t)27 * a.co * ci;
    const int nchunk = (a.npts + kWgChunk - 1) / kWgChunk;
    wg_add(P, a, blocks((size_t)a.npad * (ci + a.co) / 8));
    wg_add(R, a, blocks(nw) + a.co);
    // two output tiles per wave share the input's loads where that leaves a wave for every CU
    const size_t tasks = (size_t)9 * (ci / 16) * (a.co / 16) * nchunk;
    const int two = a.co % 32 == 0 && tasks / 2 >= 256;
    const int g = a.nx % 8 == 0 ? 3 : a.nx % 4 == 0 ? 2 : a.nx % 2 == 0 ? 1 : 0;
    wg_add(W[two][g], a, two ? tasks / 2 : tasks);
  }
  hipLaunchKernelGGL(k_wg_pack, dim3(P.off[P.n]), dim3(256), 0, u->stream, P);
  ULAUNCH("k_wg_pack");
#define WG_LAUNCH(two, g, G)                                                                                           \
  if (W[two][g].n) {                                                                                                   \
    hipLaunchKernelGGL((k_wgrad<two + 1, G>), dim3(W[two][g].off[W[two][g].n]), dim3(64), 0, u->stream, W[two][g]);     \
    ULAUNCH("k_wgrad");                                                                                                \
  }
  WG_LAUNCH(0, 3, 8) WG_LAUNCH(0, 2, 4) WG_LAUNCH(0, 1, 2) WG_LAUNCH(0, 0, 1)
  WG_LAUNCH(1, 3, 8) WG_LAUNCH(1, 2, 4) WG_LAUNCH(1, 1, 2) WG_LAUNCH(1, 0, 1)
#undef WG_LAUNCH
  hipLaunchKernelGGL(k_wg_reduce, dim3(R.off[R.n]), dim3(256), 0, u->stream, R);
  ULAUNCH("k_wg_reduce");
  return 0;
}

// data gradient of conv layer l's input ([np][c1 + c2]): FP32 into fx, or masked by the activation into gn
int layer_dgrad(salmon_unet *u, const Layer &l, const bf16_t *g, float *fx, bf16_t *gn = nullptr,
                const bf16_t *mask = nullptr) {
  const int ci = l.c1 + l.c2;
  return launch_conv(u, g, l.co, 0, nullptr, 0, l.wb, nullptr, ci, 0, l.level, gn, fx, mask);
}

int backward(salmon_unet *u, const float *target, float *loss) {
  const size_t n0 = u->np[0];
  const unsigned nb0 = blocks(n0);
  hipLaunchKernelGGL(k_mse, dim3(nb0), dim3(256), 0, u->stream, u->d_out, target, n0, u->d_dout, u->d_part);
  ULAUNCH("k_mse");
  if (loss) {
    hipLaunchKernelGGL(k_loss, dim3(1), dim3(256), 0, u->stream, u->d_part, (int)nb0, n0, loss);
    ULAUNCH("k_loss");
  }
  hipLaunchKernelGGL(k_head_grad, dim3(5), dim3(256), 0, u->stream, u->d_dout, u->act[D1B], n0, u->d_g + u->head_off);
  ULAUNCH("k_head_grad");
  hipLaunchKernelGGL(k_head_back, dim3(blocks(n0 * 16)), dim3(256), 0, u->stream, u->d_dout, u->d_w + u->head_off,
                     u->act[D1B], n0, u->g[9]);
  ULAUNCH("k_head_back");
  // conv layers in reverse; layer index li <-> act index
  static const int conv_act[10] = {E1A, E1B, E2A, E2B, E3A, E3B, D2A, D2B, D1A, D1B};
  for (int li = 9; li >= 0; --li) {
    const Layer &l = u->L[li];
    const int i = conv_act[li];
    if (li == 0) break;
    const bf16_t *g = u->g[li];
    bf16_t *gn = u->g[li - 1];
    // the gradients of D1A's and D2A's inputs are kept for their skip parts (fx is reused by the next layers)
    float *fx = i == D1A ? u->d_fx + u->fx_n : i == D2A ? u->d_fx + u->fx_n + n0 * 48 : u->d_fx;
    const bool chain = i == D1B || i == D2B || i == E3B || i == E2B || i == E1B;  // input is the previous activation
    if (int rc = chain ? layer_dgrad(u, l, g, nullptr, gn, u->act[i - 1]) : layer_dgrad(u, l, g, fx)) return rc;
    const int lv = l.level;
    const int ci = l.c1 + l.c2;
    switch (i) {
      case D1B: case D2B: case E3B: case E2B: case E1B:
        break;
      case D1A: case D2A: {
        // input [up(d2b | e3b), e1b | e2b]: the up part goes to the coarse activation, the skip part is kept
        const int up = i == D1A ? D2B : E3B;
        const int C1 = l.c1;
        hipLaunchKernelGGL(k_downsum, dim3(blocks(u->np[lv + 1] * C1)), dim3(256), 0, u->stream, fx, ci, C1,
                           u->act[up], gn, u->n[lv + 1][0], u->n[lv + 1][1], u->n[lv + 1][2]);
        ULAUNCH("k_downsum");
        break;
      }
      case E3A: case E2A: {
        // input is a pooled tensor: gradient goes back through the pool into e2b | e1b, plus the skip part
        const int dst = i == E3A ? E2B : E1B;
        const int lvf = lv - 1;
        const int Cs = i == E3A ? 96 : 48;
        const int off = i == E3A ? 64 : 32;
        const float *skip = i == E3A ? u->d_fx + u->fx_n + n0 * 48 : u->d_fx + u->fx_n;
        hipLaunchKernelGGL(k_poolback, dim3(blocks(u->np[lvf] * ci)), dim3(256), 0, u->stream, u->d_fx, skip, Cs, off,
                           ci, u->act[dst], u->n[lvf][0], u->n[lvf][1], u->n[lvf][2], gn);
        ULAUNCH("k_poolback");
        break;
      }
      default:
        return ufail(SALMON_HIP_EINVAL, "internal: layer %d", i);
    }
  }
  return weight_grads(u, conv_act);
}

int ucheck(salmon_unet_t u) { return u ? 0 : ufail(SALMON_HIP_EINVAL, "null predictor handle"); }

}  // namespace

extern "C" {

int salmon_unet_create(int nx, int ny, int nz, unsigned long long seed, salmon_unet_t *out) {
  if (!out) return ufail(SALMON_HIP_EINVAL, "out is null");
  *out = nullptr;
  if (nx % 4 || ny % 4 || nz % 4 || nx < 8 || ny < 8 || nz < 8)
    return ufail(SALMON_HIP_EUNSUPPORTED, "grid %dx%dx%d: extents must be multiples of 4, >= 8", nx, ny, nz);
  salmon_unet *u = new salmon_unet();
  for (int lv = 0; lv < 3; ++lv) {
    u->n[lv][0] = nx >> lv; u->n[lv][1] = ny >> lv; u->n[lv][2] = nz >> lv;
    u->np[lv] = (size_t)u->n[lv][0] * u->n[lv][1] * u->n[lv][2];
  }
  // conv layers: co, c1, c2, up1, level
  const int spec[10][5] = {{16, 16, 0, 0, 0}, {16, 16, 0, 0, 0}, {32, 16, 0, 0, 1}, {32, 32, 0, 0, 1},
                           {64, 32, 0, 0, 2}, {64, 64, 0, 0, 2}, {32, 64, 32, 1, 1}, {32, 32, 0, 0, 1},
                           {16, 32, 16, 1, 0}, {16, 16, 0, 0, 0}};
  size_t off = 0;
  for (auto &sp : spec) {
    Layer l;
    l.co = sp[0]; l.c1 = sp[1]; l.c2 = sp[2]; l.up1 = sp[3]; l.level = sp[4];
    l.woff = off;
    off += (size_t)27 * l.co * (l.c1 + l.c2);
    l.boff = off;
    off += l.co;
    u->L.push_back(l);
  }
  u->head_off = off;
  off += 17;
  u->nparam = off;
  auto bail = [&](int rc) { salmon_unet_destroy(u); return rc; };
  int rc;
  if ((rc = ualloc(u, &u->d_w, off)) || (rc = ualloc(u, &u->d_g, off)) || (rc = ualloc(u, &u->d_m, off)) ||
      (rc = ualloc(u, &u->d_v, off)))
    return bail(rc);
  for (Layer &l : u->L) {
    const size_t nw = (size_t)27 * l.co * (l.c1 + l.c2);
    if ((rc = ualloc(u, &l.wt, nw)) || (rc = ualloc(u, &l.wb, nw))) return bail(rc);
  }
  const size_t n0 = u->np[0], n1 = u->np[1], n2 = u->np[2];
  const size_t act_n[12] = {n0 * 16, n0 * 16, n1 * 16, n1 * 32, n1 * 32, n2 * 32, n2 * 64, n2 * 64,
                            n1 * 32, n1 * 32, n0 * 16, n0 * 16};
  if ((rc = ualloc(u, &u->x0, n0 * 16)) || (rc = ualloc(u, &u->d_zero, kConvZero))) return bail(rc);
  for (int i = 0; i < 12; ++i)
    if ((rc = ualloc(u, &u->act[i], act_n[i]))) return bail(rc);
  // d_fx: data gradient (max np * ci) followed by the two kept skip gradients (n0 x 48, n1 x 96)
  u->fx_n = std::max({n0 * 48, n1 * 96, n2 * 64, n1 * 32, n0 * 16});
  size_t wp = 0, xt = 0, gt = 0, gl = 0;
  for (Layer &l : u->L) {
    const size_t ci = l.c1 + l.c2, np = u->np[l.level];
    l.part_off = wp;
    l.xt_off = xt;
    l.gt_off = gt;
    wp += (np + kWgChunk - 1) / kWgChunk * 27 * l.co * ci;
    xt += 3 * ci * wg_pad(np);
    gt += l.co * wg_pad(np);
    gl += l.co * np;
  }
  const size_t fx_all = u->fx_n + n0 * 48 + n1 * 96;
  float *data, *grad;
  if ((rc = ualloc(u, &u->d_out, n0)) || (rc = ualloc(u, &u->d_dout, n0)) || (rc = ualloc(u, &u->d_part, blocks(n0))) ||
      (rc = ualloc(u, &data, std::max(fx_all, (xt + 1) / 2))) || (rc = ualloc(u, &grad, std::max(wp, (gl + 1) / 2))) ||
      (rc = ualloc(u, &u->d_gt, gt)) || (rc = ualloc(u, &u->d_rpart, 1024)))
    return bail(rc);
  u->d_fx = data;
  u->d_xt = (bf16_t *)data;
  u->d_wpart = grad;
  gl = 0;
  for (int li = 0; li < 10; ++li) {  // (each a whole number of 32 bytes: co is a multiple of 16)
    u->g[li] = (bf16_t *)grad + gl;
    gl += u->np[u->L[li].level] * u->L[li].co;
  }
  // He-normal weights, zero biases; head: small normal weights, zero bias
  std::vector<float> w(off, 0.f);
  std::mt19937_64 gen(seed);
  for (Layer &l : u->L) {
    const int fan_in = 27 * (l.c1 + l.c2);
    std::normal_distribution<float> nd(0.f, std::sqrt(2.f / fan_in));
    for (size_t k = 0; k < (size_t)27 * l.co * (l.c1 + l.c2); ++k) w[l.woff + k] = nd(gen);
  }
  std::normal_distribution<float> nh(0.f, 0.25f);
  for (int c = 0; c < 16; ++c) w[u->head_off + c] = nh(gen);
  if (hipMemcpy(u->d_w, w.data(), sizeof(float) * off, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemset(u->d_g, 0, sizeof(float) * off) != hipSuccess || hipMemset(u->d_m, 0, sizeof(float) * off) != hipSuccess ||
      hipMemset(u->d_v, 0, sizeof(float) * off) != hipSuccess || hipMemset(u->x0, 0, sizeof(bf16_t) * n0 * 16) != hipSuccess ||
      hipMemset(u->d_zero, 0, sizeof(bf16_t) * kConvZero) != hipSuccess)
    return bail(ufail(SALMON_HIP_EHIP, "predictor initialisation copies failed"));
  *out = u;
  return 0;
}

int salmon_unet_destroy(salmon_unet_t u) {
  if (!u) return 0;
  if (u->stream) (void)hipStreamSynchronize(u->stream);
  else (void)hipDeviceSynchronize();
  for (void *p : u->allocs) (void)hipFree(p);
  delete u;
  return 0;
}

int salmon_unet_set_stream(salmon_unet_t u, void *stream) {
  if (int rc = ucheck(u)) return rc;
  u->stream = (hipStream_t)stream;
  return 0;
}

int salmon_unet_num_params(salmon_unet_t u, long *n) {
  if (int rc = ucheck(u)) return rc;
  if (!n) return ufail(SALMON_HIP_EINVAL, "null pointer");
  *n = (long)u->nparam;
  return 0;
}

int salmon_unet_get_params(salmon_unet_t u, float *host) {
  if (int rc = ucheck(u)) return rc;
  if (!host) return ufail(SALMON_HIP_EINVAL, "null pointer");
  UHIP(hipMemcpyAsync(host, u->d_w, sizeof(float) * u->nparam, hipMemcpyDeviceToHost, u->stream));
  UHIP(hipStreamSynchronize(u->stream));
  return 0;
}

int salmon_unet_set_params(salmon_unet_t u, const float *host) {
  if (int rc = ucheck(u)) return rc;
  if (!host) return ufail(SALMON_HIP_EINVAL, "null pointer");
  UHIP(hipMemcpyAsync(u->d_w, host, sizeof(float) * u->nparam, hipMemcpyHostToDevice, u->stream));
  UHIP(hipStreamSynchronize(u->stream));
  u->packed = false;
  return 0;
}

int salmon_unet_get_grads(salmon_unet_t u, float *host) {
  if (int rc = ucheck(u)) return rc;
  if (!host) return ufail(SALMON_HIP_EINVAL, "null pointer");
  UHIP(hipMemcpyAsync(host, u->d_g, sizeof(float) * u->nparam, hipMemcpyDeviceToHost, u->stream));
  UHIP(hipStreamSynchronize(u->stream));
  return 0;
}

int salmon_unet_get_activation(salmon_unet_t u, int index, float *host, long n) {
  if (int rc = ucheck(u)) return rc;
  if (!host || index < -1 || index >= 12) return ufail(SALMON_HIP_EINVAL, "activation %d", index);
  static const int ch[12] = {16, 16, 16, 32, 32, 32, 64, 64, 32, 32, 16, 16};
  static const int lv[12] = {0, 0, 1, 1, 1, 2, 2, 2, 1, 1, 0, 0};
  const size_t cnt = index < 0 ? u->np[0] * 16 : u->np[lv[index]] * ch[index];
  if ((size_t)n != cnt) return ufail(SALMON_HIP_EINVAL, "activation %d has %zu values, not %ld", index, cnt, n);
  std::vector<bf16_t> tmp(cnt);
  UHIP(hipMemcpyAsync(tmp.data(), index < 0 ? u->x0 : u->act[index], sizeof(bf16_t) * cnt, hipMemcpyDeviceToHost,
                      u->stream));
  UHIP(hipStreamSynchronize(u->stream));
  for (size_t i = 0; i < cnt; ++i) {
    const unsigned v = (unsigned)tmp[i] << 16;
    memcpy(host + i, &v, 4);
  }
  return 0;
}

int salmon_unet_forward(salmon_unet_t u, const float *in_dev, float *out_dev) {
  if (int rc = ucheck(u)) return rc;
  if (!in_dev || !out_dev) return ufail(SALMON_HIP_EINVAL, "null pointer");
  return forward(u, in_dev, out_dev);
}

int salmon_unet_train_sample(salmon_unet_t u, const float *in_dev, const float *target_dev, float *loss_dev) {
  if (int rc = ucheck(u)) return rc;
  if (!in_dev || !target_dev) return ufail(SALMON_HIP_EINVAL, "null pointer");
  if (int rc = forward(u, in_dev, u->d_out)) return rc;
  return backward(u, target_dev, loss_dev);
}

int salmon_unet_features(salmon_unet_t u, const double *v0, const double *v1, const double *v2, const double *v3,
                         const double *vpsl, double s_diff, double s_abs, float *in_dev) {
  if (int rc = ucheck(u)) return rc;
  if (!v0 || !v1 || !v2 || !v3 || !vpsl || !in_dev) return ufail(SALMON_HIP_EINVAL, "null pointer");
  if (!(s_diff > 0.0) || !(s_abs > 0.0)) return ufail(SALMON_HIP_EINVAL, "scales must be positive");
  hipLaunchKernelGGL(k_features, dim3(blocks(u->np[0])), dim3(256), 0, u->stream, v0, v1, v2, v3, vpsl, s_diff, s_abs,
                     u->np[0], in_dev);
  ULAUNCH("k_features");
  return 0;
}

int salmon_unet_predict(salmon_unet_t u, const double *v0, const double *v1, const float *nn_dev, double s_out,
                        double *vpred_dev) {
  if (int rc = ucheck(u)) return rc;
  if (!v0 || !v1 || !nn_dev || !vpred_dev) return ufail(SALMON_HIP_EINVAL, "null pointer");
  hipLaunchKernelGGL(k_predict, dim3(blocks(u->np[0])), dim3(256), 0, u->stream, v0, v1, nn_dev, s_out, u->np[0],
                     vpred_dev);
  ULAUNCH("k_predict");
  return 0;
}

int salmon_unet_target(salmon_unet_t u, const double *vmid, const double *v0, const double *v1, double s_out,
                       float *t_dev) {
  if (int rc = ucheck(u)) return rc;
  if (!vmid || !v0 || !v1 || !t_dev) return ufail(SALMON_HIP_EINVAL, "null pointer");
  if (!(s_out > 0.0)) return ufail(SALMON_HIP_EINVAL, "scale must be positive");
  hipLaunchKernelGGL(k_target, dim3(blocks(u->np[0])), dim3(256), 0, u->stream, vmid, v0, v1, s_out, u->np[0], t_dev);
  ULAUNCH("k_target");
  return 0;
}

int salmon_unet_residual(salmon_unet_t u, const double *vpred, const double *v0, const double *vnew, double *out_dev) {
  if (int rc = ucheck(u)) return rc;
  if (!vpred || !v0 || !vnew || !out_dev) return ufail(SALMON_HIP_EINVAL, "null pointer");
  const int nb = (int)std::min<size_t>(1024, blocks(u->np[0]));
  hipLaunchKernelGGL(k_resid_part, dim3(nb), dim3(256), 0, u->stream, vpred, v0, vnew, u->np[0], u->d_rpart);
  ULAUNCH("k_resid_part");
  hipLaunchKernelGGL(k_resid_final, dim3(1), dim3(256), 0, u->stream, u->d_rpart, nb, out_dev);
  ULAUNCH("k_resid_final");
  return 0;
}

int salmon_unet_gate(salmon_unet_t u, const double *resid_dev, double tol, int *flag_dev, int *stats_dev,
                     double *log_dev, int log_cap) {
  if (int rc = ucheck(u)) return rc;
  if (!resid_dev || !flag_dev || !stats_dev || (log_cap > 0 && !log_dev))
    return ufail(SALMON_HIP_EINVAL, "null pointer");
  hipLaunchKernelGGL(k_gate, dim3(1), dim3(64), 0, u->stream, resid_dev, tol, flag_dev, stats_dev,
                     log_cap > 0 ? log_dev : nullptr, log_cap);
  ULAUNCH("k_gate");
  return 0;
}

int salmon_unet_adam_step(salmon_unet_t u, float lr, int nsamples) {
  if (int rc = ucheck(u)) return rc;
  if (nsamples < 1) return ufail(SALMON_HIP_EINVAL, "nsamples=%d", nsamples);
  u->adam_t += 1;
  const float c1 = 1.f - std::pow(0.9f, (float)u->adam_t);
  const float c2 = 1.f - std::pow(0.999f, (float)u->adam_t);
  hipLaunchKernelGGL(k_adam, dim3(blocks(u->nparam)), dim3(256), 0, u->stream, u->nparam, u->d_w, u->d_g, u->d_m,
                     u->d_v, lr, c1, c2, 1.f / (float)nsamples);
  ULAUNCH("k_adam");
  u->packed = false;
  return 0;
}

}  // extern "C"
