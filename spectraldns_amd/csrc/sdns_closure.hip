// Learned subgrid closure kernels (declared in sdns_closure.hpp).
//
// The 3x3x3 periodic convolution is an implicit GEMM on the bf16 matrix cores:
// v_mfma_f32_16x16x32_bf16 multiplies A (16 x 32) by B (32 x 16) into a 16 x 16
// FP32 tile.  Lane l (0..63) holds A[l % 16][8 (l / 16) + j], B[8 (l / 16) + j][l % 16]
// (j = 0..7) and D[4 (l / 16) + i][l % 16] (i = 0..3).  In the forward
// product A rows are output channels, K is the input channel index (32
// channels per tap, or 4 taps x 8 channels for 8-channel inputs) and B columns
// are 16 consecutive points of one z-row; channels-last storage makes every A
// and B fragment one 16-byte load per lane.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "sdns_closure.hpp"

namespace sdns {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float silu_f(float z) { return z / (1.0f + expf(-z)); }
__device__ __forceinline__ float dsilu_f(float z) {
  const float s = 1.0f / (1.0f + expf(-z));
  return s * (1.0f + z * (1.0f - s));
}
__device__ __forceinline__ int wrap(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

// ------------------------------------------------------------------ convolution
// Both kernels multiply the weights as the A operand (rows = 16 output
// channels) with 16 consecutive points of one z-row as the B operand, so a lane
// ends with D[4 g + i][m] = channels 16 b + 4 g + i of point m: four adjacent
// channels, one 8-byte (bf16) or 16-byte (FP32) access each in the epilogue.
// With the operands the other way round a lane held four points of one
// channel and the epilogue's 2-byte accesses took as long as the products
// (64^3: layer 2 43 us, its input gradient 59 us).
template <int EPI, int COUT>
__device__ __forceinline__ void conv_epilogue(const ConvArgs& a, const f32x4& acc, const f32x4& bias, long pt, int co) {
  f32x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = acc[i] + bias[i];
  if constexpr (EPI == CONV_EPI_SILU) {
    bf16x4 z, r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      z[i] = (__bf16)v[i];
      r[i] = (__bf16)silu_f((float)z[i]);
    }
    if (a.z) *(bf16x4*)(a.z + pt * COUT + co) = z;
    *(bf16x4*)(a.a + pt * COUT + co) = r;
  } else if constexpr (EPI == CONV_EPI_DSILU) {
    const bf16x4 z = *(const bf16x4*)(a.zprev + pt * COUT + co);
    bf16x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = (__bf16)(v[i] * dsilu_f((float)z[i]));
    *(bf16x4*)(a.a + pt * COUT + co) = r;
  } else if constexpr (EPI == CONV_EPI_PLANAR) {
    const long P = (long)a.n0 * a.n1 * a.n2;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (co + i < a.ncout) a.y[(co + i) * P + pt] = v[i] * a.scale;
  } else {
    float* y = a.y + pt * a.ystride + co;
    if (co + 4 <= a.ncout) {
      *(f32x4*)y = v;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (co + i < a.ncout) y[i] = v[i];
    }
  }
}
template <int EPI> __device__ __forceinline__ f32x4 conv_bias(const ConvArgs& a, int co) {
  return a.bias ? *(const f32x4*)(a.bias + co) : f32x4{0.f, 0.f, 0.f, 0.f};
}

// 8-channel inputs: K = 32 is 4 taps x 8 channels, seven K-steps (k-group g of
// step s is tap 4 s + g; the 28th tap is zeros).  A block owns 4 y-rows x 16 MT z
// points of two x-planes and stages their halo (4 planes x 6 rows x (16 MT + 2)
// points of 16 bytes, 25 KB) in LDS; wave w computes row w of both planes with
// the layer's weights in registers.  (Fragments straight from global memory,
// 7 KB per 16 points through L1, took 19 us at 64^3.)
constexpr int CONV8_XP = 2, CONV_ROWS = 4;
// PLANAR: the input is the planar FP32 velocity, scaled and rounded to bf16 as it
// is staged (inference; training keeps the packed input for its weight gradient):
// with the six stress components transformed together, 234 -> 228 us an LES step
// at 64^3.
template <int COUT, int EPI, int MT, bool PLANAR>
__global__ void __launch_bounds__(256) k_conv8(ConvArgs a) {
  constexpr int NB = COUT / 16, KS = 7, npt = 16 * MT + 2;
  constexpr int PC = (CONV_ROWS + 2) * npt, NC = (CONV8_XP + 2) * PC, NR = (NC + 255) / 256;
  __shared__ bf16x8 hl[NC];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int m = lane & 15, g = lane >> 4;
  const int n0 = a.n0, n1 = a.n1, n2 = a.n2;
  const int nzb = n2 / (16 * MT), nrb = (n1 + CONV_ROWS - 1) / CONV_ROWS;
  int blk = blockIdx.x;
  const int z0 = blk % nzb * (16 * MT);
  blk /= nzb;
  const int i1b = blk % nrb * CONV_ROWS, x0 = blk / nrb * CONV8_XP;
  const bf16x8* __restrict__ X = (const bf16x8*)a.x;
  const bf16x8* __restrict__ W = (const bf16x8*)a.w;
  bf16x8 r[NR];
#pragma unroll
  for (int e = 0; e < NR; ++e) {
    const int c = min((int)threadIdx.x + 256 * e, NC - 1);
    const int pt = c % npt, row = c / npt % (CONV_ROWS + 2), j = c / PC;
    const long q = ((long)wrap(x0 + j - 1, n0) * n1 + wrap(i1b + row - 1, n1)) * n2 + wrap(z0 + pt - 1, n2);
    if constexpr (PLANAR) {
      const long P = (long)n0 * n1 * n2;
      r[e] = bf16x8{};
#pragma unroll
      for (int ch = 0; ch < 3; ++ch) r[e][ch] = (__bf16)(a.u[ch * P + q] * a.scale);
    } else {
      r[e] = X[q];
    }
  }
  bf16x8 wv[KS][NB];
  int off[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int tap = 4 * s + g < 27 ? 4 * s + g : 26;
#pragma unroll
    for (int b = 0; b < NB; ++b) wv[s][b] = 4 * s + g < 27 ? W[tap * COUT + b * 16 + m] : bf16x8{};
    off[s] = (tap / 9) * PC + (w + tap / 3 % 3) * npt + tap % 3 + m;
  }
  f32x4 bias[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) bias[b] = conv_bias<EPI>(a, 16 * b + 4 * g);
#pragma unroll
  for (int e = 0; e < NR; ++e)
    if (threadIdx.x + 256 * e < NC) hl[threadIdx.x + 256 * e] = r[e];
  __syncthreads();
  if (i1b + w >= n1) return;
  for (int k = 0; k < CONV8_XP && x0 + k < n0; ++k) {
    const long prow = ((long)(x0 + k) * n1 + i1b + w) * n2 + z0;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      f32x4 acc[NB];
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        bf16x8 pv = hl[k * PC + off[s] + 16 * t];
        if (s == KS - 1 && 4 * s + g >= 27) pv = bf16x8{};
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[s][b], pv, acc[b], 0, 0, 0);
      }
#pragma unroll
      for (int b = 0; b < NB; ++b) conv_epilogue<EPI, COUT>(a, acc[b], bias[b], prow + 16 * t + m, 16 * b + 4 * g);
    }
  }
}

// 32-channel inputs, LDS-tiled.  A block owns 4 consecutive y-rows x 16 MT
// consecutive z points over CONV_XP consecutive x-planes, and marches along
// x: the layer's weights (all 27 taps) stay in LDS, and the periodic input
// halo is a rolling window of x-planes (6 rows x (16 MT + 2) points each) in 4
// LDS slots, the plane after next loaded into registers while the current
// output plane is computed and stored into its free slot afterwards.  One
// block fills a CU's LDS (157 KB at 32 -> 32 channels and 64 points), so it has
// 8 waves: waves w and w + 4 compute the two halves of row w, and each wave
// finishes a plane (SiLU is about 40 VALU instructions a value, more time than
// the products) between the next plane's products, the two waves of a SIMD at
// different taps.  Rows and planes past the grid are computed
// from wrapped input and not stored.
constexpr int CONV_XP = 4, CONV_SLOTS = 4;
template <int COUT> constexpr int conv_w_bytes() { return 27 * COUT * 32 * 2; }
constexpr int conv_plane_chunks(int tzn) { return (CONV_ROWS + 2) * (tzn + 2) * 4; }

template <int COUT, int EPI, int MT>
__global__ void __launch_bounds__(512, 2) k_conv_lds(ConvArgs a) {
  constexpr int NB = COUT / 16, MW = MT / 2;
  constexpr int tzn = 16 * MT, npt = tzn + 2, PC = conv_plane_chunks(tzn);
  constexpr int PR = (PC + 511) / 512;  // prefetch registers (16-byte chunks) per thread
  extern __shared__ __align__(16) unsigned char conv_smem[];
  bf16x8* wl = (bf16x8*)conv_smem;
  bf16x8* hl = (bf16x8*)(conv_smem + conv_w_bytes<COUT>());
  const int n0 = a.n0, n1 = a.n1, n2 = a.n2;
  const int nzb = n2 / tzn, nrb = (n1 + CONV_ROWS - 1) / CONV_ROWS;
  int blk = blockIdx.x;
  const int zb = blk % nzb;
  blk /= nzb;
  const int rb = blk % nrb, xc = blk / nrb;
  const int i1b = rb * CONV_ROWS, z0 = zb * tzn, x0 = xc * CONV_XP;
  const int nx = min(CONV_XP, n0 - x0);
  const bf16x8* __restrict__ X = (const bf16x8*)a.x;
  const bf16x8* __restrict__ W = (const bf16x8*)a.w;
  // chunk c of an input plane: (row, point, channel group), row-major
  int coff[PR];
#pragma unroll
  for (int e = 0; e < PR; ++e) {
    const int c = threadIdx.x + 512 * e;
    const int cg = c % 4, q = c / 4, pt = q % npt, row = q / npt;
    coff[e] = (wrap(i1b + row - 1, n1) * n2 + wrap(z0 + pt - 1, n2)) * 4 + cg;
  }
  auto load_plane = [&](int j, bf16x8 (&r)[PR]) {
    const bf16x8* p = X + (long)wrap(x0 + j, n0) * n1 * n2 * 4;
#pragma unroll
    for (int e = 0; e < PR; ++e)
      if (threadIdx.x + 512 * e < PC) r[e] = p[coff[e]];
  };
  auto store_plane = [&](int j, const bf16x8 (&r)[PR]) {
    bf16x8* dst = hl + ((j + 1) % CONV_SLOTS) * PC;
#pragma unroll
    for (int e = 0; e < PR; ++e)
      if (threadIdx.x + 512 * e < PC) dst[threadIdx.x + 512 * e] = r[e];
  };
  bf16x8 pre[PR], p0[PR], p1[PR];
  load_plane(-1, p0);  // planes x0 - 1, x0, x0 + 1
  load_plane(0, p1);
  load_plane(1, pre);
  constexpr int WC = 27 * COUT * 4, WR = (WC + 511) / 512;
  bf16x8 wr[WR];
#pragma unroll
  for (int e = 0; e < WR; ++e) wr[e] = W[min((int)threadIdx.x + 512 * e, WC - 1)];
#pragma unroll
  for (int e = 0; e < WR; ++e)
    if (threadIdx.x + 512 * e < WC) wl[threadIdx.x + 512 * e] = wr[e];
  store_plane(-1, p0);
  store_plane(0, p1);
  store_plane(1, pre);
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int w = wave & 3, half = wave >> 2;
  const int m = lane & 15, g = lane >> 4;
  const bool row_ok = i1b + w < n1;
  f32x4 bias[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) bias[b] = conv_bias<EPI>(a, 16 * b + 4 * g);
  f32x4 acc[MW][NB], done[MW][NB];  // this plane's sums, the last plane's
  auto finish = [&](int k, int i) {
    const long prow = ((long)(x0 + k) * n1 + i1b + w) * n2 + z0;
    const int t = i / NB, b = i % NB;
    conv_epilogue<EPI, COUT>(a, done[t][b], bias[b], prow + 16 * (half * MW + t) + m, 16 * b + 4 * g);
  };
  for (int k = 0; k < nx; ++k) {
    const bool more = k + 1 < nx, pending = k > 0 && row_ok;
    if (more) load_plane(k + 2, pre);  // in flight during this plane's products
    const bf16x8* const pl[3] = {hl + (k % CONV_SLOTS) * PC, hl + ((k + 1) % CONV_SLOTS) * PC,
                                 hl + ((k + 2) % CONV_SLOTS) * PC};
#pragma unroll
    for (int t = 0; t < MW; ++t)
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[t][b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int tap = 0; tap < 27; ++tap) {
      const int tz = tap / 9, ty = (tap / 3) % 3, tx = tap % 3;
      bf16x8 wv[NB], pv[MW];
#pragma unroll
      for (int b = 0; b < NB; ++b) wv[b] = wl[(tap * COUT + b * 16 + m) * 4 + g];
      const bf16x8* h = pl[tz] + ((w + ty) * npt + half * MW * 16 + m + tx) * 4 + g;
#pragma unroll
      for (int t = 0; t < MW; ++t) pv[t] = h[64 * t];
#pragma unroll
      for (int t = 0; t < MW; ++t)
#pragma unroll
        for (int b = 0; b < NB; ++b)
          acc[t][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[b], pv[t], acc[t][b], 0, 0, 0);
      // the last plane's epilogue, a fragment every third tap: waves 0..3 in the
      // first half of the taps, waves 4..7 in the second
      if (tap % 3 == 2 && tap / 3 < MW * NB) {
        if (pending && half == 0) finish(k - 1, tap / 3);
      }
      if (tap % 3 == 2 && tap / 3 >= 4 && tap / 3 - 4 < MW * NB) {
        if (pending && half == 1) finish(k - 1, tap / 3 - 4);
      }
    }
#pragma unroll
    for (int t = 0; t < MW; ++t)
#pragma unroll
      for (int b = 0; b < NB; ++b) done[t][b] = acc[t][b];
    // the slot of plane k + 2 held plane k - 2, which no wave reads any more
    if (more) {
      store_plane(k + 2, pre);
      __syncthreads();
    }
  }
  if (row_ok) {
#pragma unroll
    for (int i = 0; i < MW * NB; ++i) finish(nx - 1, i);
  }
}

template <int COUT, int EPI, int MT> int conv_lds_go(const ConvArgs& a, hipStream_t s) {
  const size_t bytes = (size_t)conv_w_bytes<COUT>() + (size_t)CONV_SLOTS * conv_plane_chunks(16 * MT) * 16;
  // dynamic LDS beyond 64 KB must be allowed for the kernel (on the current device)
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(&k_conv_lds<COUT, EPI, MT>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess)
    return -1;
  const long nblk = (long)((a.n0 + CONV_XP - 1) / CONV_XP) * ((a.n1 + CONV_ROWS - 1) / CONV_ROWS) * (a.n2 / (16 * MT));
  hipLaunchKernelGGL((k_conv_lds<COUT, EPI, MT>), dim3((unsigned)nblk), dim3(512), bytes, s, a);
  return 0;
}
template <int CIN, int COUT, int EPI, int MT> int conv_go(const ConvArgs& a, hipStream_t s) {
  if constexpr (CIN == 32) {
    return conv_lds_go<COUT, EPI, MT>(a, s);
  } else {
    const long nblk =
        (long)((a.n0 + CONV8_XP - 1) / CONV8_XP) * ((a.n1 + CONV_ROWS - 1) / CONV_ROWS) * (a.n2 / (16 * MT));
    if constexpr (EPI == CONV_EPI_SILU)
      if (!a.x) {
        hipLaunchKernelGGL((k_conv8<COUT, EPI, MT, true>), dim3((unsigned)nblk), dim3(256), 0, s, a);
        return 0;
      }
    hipLaunchKernelGGL((k_conv8<COUT, EPI, MT, false>), dim3((unsigned)nblk), dim3(256), 0, s, a);
    return 0;
  }
}

int launch_conv(int cin, int cout, int epi, const ConvArgs& a, hipStream_t s) {
  if (a.n2 % 32 || a.n0 < 4 || a.n1 < 4) return -1;
#define SDNS_CONV(CI, CO, EP)                                                                       \
  if (cin == CI && cout == CO && epi == EP)                                                         \
    return a.n2 % 64 ? conv_go<CI, CO, EP, 2>(a, s) : conv_go<CI, CO, EP, 4>(a, s);
  SDNS_CONV(8, 32, CONV_EPI_SILU)      // layer 1 forward
  SDNS_CONV(32, 32, CONV_EPI_SILU)     // layer 2 forward
  SDNS_CONV(32, 16, CONV_EPI_LINEAR)   // layer 3 forward (training)
  SDNS_CONV(32, 16, CONV_EPI_PLANAR)   // layer 3 forward (inference)
  SDNS_CONV(8, 32, CONV_EPI_DSILU)     // layer 3 input gradient -> layer 2 pre-activation gradient
  SDNS_CONV(32, 32, CONV_EPI_DSILU)    // layer 2 input gradient -> layer 1 pre-activation gradient
#undef SDNS_CONV
  return -1;
}

// ------------------------------------------------------------------ weight gradient
// dW[tap][co][ci] = sum_p g[p][co] x[p + d(tap)][ci]: M = co, N = ci, K = points.
// The fields are channels-last, so a fragment's 8 consecutive points of one
// channel are 8 rows apart; they are read from LDS with the transposing
// 4 x 16 read (ds_read_b64_tr_b16: lane j of 16 supplies the address of row
// j / 4, columns 4 (j % 4).., and receives column j of the four rows).  A block
// owns 4 y-rows x TZ z points of up to WG_XP x-planes and one of the three x
// offsets of the taps (blockIdx.y): it stages g (4 rows) and x (6 rows, TZ + 2
// points) of a plane, loads the next plane into registers meanwhile, and wave w
// multiplies row w with the nine shifted rows, 32 points per product.  Every
// value is read from memory 3 times and from LDS 9 times; gathering the
// fragments from global memory with 2-byte loads, once per tap, took 73-90 us
// per layer at 64^3.  The bias gradient is one more product with ones (in the
// blocks of the middle offset).  Each block writes its sums in fragment order:
// part[set][27][WG_FR] then WG_BIAS bias sums per set.
constexpr int WG_ROWS = 4, WG_XP = 8;
template <int C> constexpr int wg_tiles() { return (C + 15) / 16; }
template <int GC, int XC> constexpr int wg_fr() { return wg_tiles<GC>() * wg_tiles<XC>() * 256; }
template <int GC, int XC> constexpr long wg_set_floats() { return 27L * wg_fr<GC, XC>() + 32; }
inline int wg_tz(int n2) { return n2 % 64 ? 32 : 64; }
inline int wg_sets(int n0, int n1, int n2) {
  return ((n0 + WG_XP - 1) / WG_XP) * ((n1 + WG_ROWS - 1) / WG_ROWS) * (n2 / wg_tz(n2));
}

// Fragment of 32 points x 16 channels from LDS rows of C channels: lane l gets
// points 8 (l / 16) .. + 7 of channel l % 16 of the tile.  Rows of 8 channels
// give tile channels 8..15 the next point's values (columns nobody uses).
template <int C> __device__ __forceinline__ bf16x8 frag_tr(const __bf16* p, int lane) {
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  const int g = lane >> 4, j = lane & 15;
  const __bf16* q = p + (8 * g + (j >> 2)) * C + 4 * (j & 3);
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)q);
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(q + 4 * C));
  typedef short s16x8 __attribute__((ext_vector_type(8)));
  const s16x8 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  return __builtin_bit_cast(bf16x8, v);
}

template <int GC, int XC, int TZ>
__global__ void __launch_bounds__(256, 2) k_wgrad(const __bf16* __restrict__ gp, const __bf16* __restrict__ xp,
                                                  float* __restrict__ part, int n0, int n1, int n2) {
  constexpr int MB = wg_tiles<GC>(), NB = wg_tiles<XC>(), FR = wg_fr<GC, XC>();
  constexpr int NPT = TZ + 2, GCH = GC / 8, XCH = XC / 8;
  constexpr int NG = WG_ROWS * TZ * GCH, NX = (WG_ROWS + 2) * NPT * XCH;  // 16-byte chunks
  constexpr int RG = (NG + 255) / 256, RX = (NX + 255) / 256;
  // (+ 2 chunks: fragments of 8-channel rows read past the last row)
  constexpr int STAGE = (NG + NX + 2) * 16, RED = 4 * MB * NB * 256 * 4;
  __shared__ __align__(16) unsigned char smem[STAGE > RED ? STAGE : RED];
  bf16x8* gs = (bf16x8*)smem;
  bf16x8* xs = gs + NG;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int nzb = n2 / TZ, nrb = (n1 + WG_ROWS - 1) / WG_ROWS;
  int blk = blockIdx.x;
  const int z0 = blk % nzb * TZ;
  blk /= nzb;
  const int i1b = blk % nrb * WG_ROWS, x0 = blk / nrb * WG_XP;
  const int nx = min(WG_XP, n0 - x0), tz = blockIdx.y;
  const bf16x8* __restrict__ G = (const bf16x8*)gp;
  const bf16x8* __restrict__ X = (const bf16x8*)xp;
  int og[RG], ox[RX];
#pragma unroll
  for (int e = 0; e < RG; ++e) {
    const int c = threadIdx.x + 256 * e, q = c / GCH, row = i1b + q / TZ;
    og[e] = c < NG && row < n1 ? (row * n2 + z0 + q % TZ) * GCH + c % GCH : -1;
  }
#pragma unroll
  for (int e = 0; e < RX; ++e) {
    const int c = threadIdx.x + 256 * e, q = c / XCH;
    ox[e] = (wrap(i1b + q / NPT - 1, n1) * n2 + wrap(z0 + q % NPT - 1, n2)) * XCH + c % XCH;
  }
  bf16x8 rg[RG], rx[RX];
  auto load = [&](int k) {
    const bf16x8* g = G + (long)(x0 + k) * n1 * n2 * GCH;
    const bf16x8* x = X + (long)wrap(x0 + k + tz - 1, n0) * n1 * n2 * XCH;
#pragma unroll
    for (int e = 0; e < RG; ++e) rg[e] = og[e] >= 0 ? g[og[e]] : bf16x8{};
#pragma unroll
    for (int e = 0; e < RX; ++e)
      if (threadIdx.x + 256 * e < NX) rx[e] = x[ox[e]];
  };
  f32x4 acc[9][MB][NB], accb[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    accb[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[t][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  bf16x8 ones;
#pragma unroll
  for (int j = 0; j < 8; ++j) ones[j] = (__bf16)1.0f;
  load(0);
  for (int k = 0; k < nx; ++k) {
#pragma unroll
    for (int e = 0; e < RG; ++e)
      if (threadIdx.x + 256 * e < NG) gs[threadIdx.x + 256 * e] = rg[e];
#pragma unroll
    for (int e = 0; e < RX; ++e)
      if (threadIdx.x + 256 * e < NX) xs[threadIdx.x + 256 * e] = rx[e];
    __syncthreads();
    if (k + 1 < nx) load(k + 1);
#pragma unroll
    for (int ks = 0; ks < TZ / 32; ++ks) {
      bf16x8 av[MB];
#pragma unroll
      for (int i = 0; i < MB; ++i) av[i] = frag_tr<GC>((const __bf16*)gs + (w * TZ + 32 * ks) * GC + 16 * i, lane);
      if (tz == 1) {
#pragma unroll
        for (int i = 0; i < MB; ++i) accb[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[i], ones, accb[i], 0, 0, 0);
      }
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        bf16x8 bv[NB];
#pragma unroll
        for (int j = 0; j < NB; ++j)
          bv[j] = frag_tr<XC>((const __bf16*)xs + ((w + t / 3) * NPT + 32 * ks + t % 3) * XC + 16 * j, lane);
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int j = 0; j < NB; ++j)
            acc[t][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[i], bv[j], acc[t][i][j], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  // sum the four waves in wave order, one tap at a time
  float* red = (float*)smem;
  float* out = part + (long)blockIdx.x * wg_set_floats<GC, XC>();
#pragma unroll
  for (int t = 0; t < 9; ++t) {
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int k = 0; k < 4; ++k) red[w * FR + ((i * NB + j) * 4 + k) * 64 + lane] = acc[t][i][j][k];
    __syncthreads();
    for (int f = threadIdx.x; f < FR; f += 256)
      out[(9 * tz + t) * FR + f] = red[f] + red[FR + f] + red[2 * FR + f] + red[3 * FR + f];
    __syncthreads();
  }
  if (tz == 1) {
    if ((lane & 15) == 0) {
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int k = 0; k < 4; ++k) red[w * 32 + 16 * i + 4 * (lane >> 4) + k] = accb[i][k];
    }
    __syncthreads();
    if (threadIdx.x < 16 * MB)
      out[27 * FR + threadIdx.x] =
          red[threadIdx.x] + red[32 + threadIdx.x] + red[64 + threadIdx.x] + red[96 + threadIdx.x];
  }
}

size_t wgrad_part_floats(int n0, int n1, int n2) {
  return (size_t)wg_sets(n0, n1, n2) * (wg_set_floats<32, 8>() + wg_set_floats<32, 32>() + wg_set_floats<8, 32>());
}
static float* wg_part(float* part, int layer, int sets) {
  return part + sets * (layer > 0 ? wg_set_floats<32, 8>() : 0) + sets * (layer > 1 ? wg_set_floats<32, 32>() : 0);
}

int launch_wgrad(int layer, const __bf16* g, const __bf16* x, float* part, int n0, int n1, int n2, hipStream_t s) {
  if (n2 % 32 || n0 < 4 || n1 < 4) return -1;
  const int sets = wg_sets(n0, n1, n2);
  const dim3 grid(sets, 3), blk(256);
  float* p = wg_part(part, layer, sets);
#define SDNS_WG(L, GC, XC)                                                                                    \
  if (layer == L) {                                                                                           \
    if (n2 % 64) hipLaunchKernelGGL((k_wgrad<GC, XC, 32>), grid, blk, 0, s, g, x, p, n0, n1, n2);             \
    else hipLaunchKernelGGL((k_wgrad<GC, XC, 64>), grid, blk, 0, s, g, x, p, n0, n1, n2);                     \
    return 0;                                                                                                 \
  }
  SDNS_WG(0, 32, 8)
  SDNS_WG(1, 32, 32)
  SDNS_WG(2, 8, 32)
#undef SDNS_WG
  return -1;
}

// All gradients from the partials in one launch, fixed order: blocks sum 64
// weight entries over the sets (four groups of sets side by side), the last
// three blocks the biases of layers 1 and 2, the bias of layer 3 (from the
// loss kernel's FP32 sums) and the loss.
constexpr int LOSS_BLOCKS = 256;
struct GradLayer {
  const float* part;
  long stride;            // floats per set
  int fr, nb;             // fragment floats per tap, ci tiles
  int cor, cir, off;      // real sizes, offset of the layer's weights in grad
  int blk0;               // first block of the layer
};
struct GradArgs {
  GradLayer l[3];
  int sets, nwblk;
  float* grad;
  const float* gsum;      // [LOSS_BLOCKS][8]
  const double* lpart;    // [LOSS_BLOCKS]
  double* loss;
  double loss_scale;
};
__global__ void __launch_bounds__(256) k_grad_reduce(GradArgs a) {
  __shared__ double sd[256];
  float* s = (float*)sd;
  const int t = threadIdx.x;
  if ((int)blockIdx.x < a.nwblk) {
    const int li = (int)blockIdx.x >= a.l[2].blk0 ? 2 : ((int)blockIdx.x >= a.l[1].blk0 ? 1 : 0);
    const GradLayer& l = a.l[li];
    const int e = ((int)blockIdx.x - l.blk0) * 64 + (t & 63), grp = t >> 6;
    const float* p = l.part + e;
    float v = 0.f;
#pragma unroll 8
    for (int b = grp; b < a.sets; b += 4) v += p[b * l.stride];
    s[t] = v;
    __syncthreads();
    if (t < 64) {
      const float sum = s[t] + s[64 + t] + s[128 + t] + s[192 + t];
      const int tap = e / l.fr, f = e % l.fr;
      const int m = f & 15, g = (f >> 4) & 3, k = (f >> 6) & 3, ij = f >> 8;
      const int co = 16 * (ij / l.nb) + 4 * g + k, ci = 16 * (ij % l.nb) + m;
      if (co < l.cor && ci < l.cir) a.grad[l.off + (tap * l.cor + co) * l.cir + ci] = sum;
    }
    return;
  }
  const int which = (int)blockIdx.x - a.nwblk;
  if (which < 3) {  // bias of layer `which`: 32 channels x 8 groups of sets
    const GradLayer& l = a.l[which];
    const int c = t & 31, grp = t >> 5;
    float v = 0.f;
    if (which < 2) {
      for (int b = grp; b < a.sets; b += 8) v += l.part[b * l.stride + 27L * l.fr + c];
    } else if (c < 8) {
      for (int b = grp; b < LOSS_BLOCKS; b += 8) v += a.gsum[b * 8 + c];
    }
    s[t] = v;
    __syncthreads();
    if (t < l.cor) {
      float sum = 0.f;
      for (int q = 0; q < 8; ++q) sum += s[32 * q + t];
      a.grad[l.off + 27 * l.cor * l.cir + t] = sum;
    }
    return;
  }
  sd[t] = a.lpart[t];
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (t < h) sd[t] += sd[t + h];
    __syncthreads();
  }
  if (t == 0 && a.loss) *a.loss = sd[0] * a.loss_scale;
}

int launch_grad_reduce(const float* part, int n0, int n1, int n2, const float* gsum, const double* lpart, float* grad,
                       double* loss, hipStream_t s) {
  GradArgs a{};
  a.sets = wg_sets(n0, n1, n2);
  const int fr[3] = {wg_fr<32, 8>(), wg_fr<32, 32>(), wg_fr<8, 32>()};
  const long st[3] = {wg_set_floats<32, 8>(), wg_set_floats<32, 32>(), wg_set_floats<8, 32>()};
  const int nb[3] = {1, 2, 2}, cor[3] = {32, 32, CL_OUT}, cir[3] = {CL_IN, 32, 32}, off[3] = {CL_OW1, CL_OW2, CL_OW3};
  int blk = 0;
  for (int l = 0; l < 3; ++l) {
    a.l[l] = {wg_part(const_cast<float*>(part), l, a.sets), st[l], fr[l], nb[l], cor[l], cir[l], off[l], blk};
    blk += 27 * fr[l] / 64;
  }
  a.nwblk = blk;
  a.grad = grad; a.gsum = gsum; a.lpart = lpart; a.loss = loss;
  a.loss_scale = 1.0 / (6.0 * (double)n0 * n1 * n2);
  hipLaunchKernelGGL(k_grad_reduce, dim3(blk + 4), dim3(256), 0, s, a);
  return 0;
}

// ------------------------------------------------------------------ loss
// Loss partials, its gradient in bf16 (pad 0) and the gradient's FP32 sums per
// channel (layer 3's bias gradient); tau planar, scaled as it is read.
__global__ void __launch_bounds__(256) k_loss(const float* __restrict__ y, const float* __restrict__ tau, float scale,
                                              __bf16* __restrict__ gyb, long n, double* __restrict__ part,
                                              float* __restrict__ gsum) {
  __shared__ double s[256];
  __shared__ float sg[4][8];
  double acc = 0.0;
  float gs[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  const float sc = 2.0f / (float)(6.0 * (double)n);
  for (long p = (long)blockIdx.x * 256 + threadIdx.x; p < n; p += (long)gridDim.x * 256) {
    bf16x8 gb = {};
    float v[8];
    *(f32x4*)v = ((const f32x4*)y)[2 * p];
    *(f32x4*)(v + 4) = ((const f32x4*)y)[2 * p + 1];
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      const float t = tau[c * n + p] * scale;
      const float d = v[c] - t;
      acc += (double)d * d;
      const float gv = sc * d;
      gs[c] += gv;
      gb[c] = (__bf16)gv;
    }
    ((bf16x8*)gyb)[p] = gb;
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int c = 0; c < 6; ++c) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) gs[c] += __shfl_down(gs[c], off, 64);
    if (lane == 0) sg[w][c] = gs[c];
  }
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) s[threadIdx.x] += s[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = s[0];
  if (threadIdx.x < 8)
    gsum[blockIdx.x * 8 + threadIdx.x] =
        threadIdx.x < 6 ? sg[0][threadIdx.x] + sg[1][threadIdx.x] + sg[2][threadIdx.x] + sg[3][threadIdx.x] : 0.f;
}
int launch_loss(const float* y, const float* tau, float scale, __bf16* gyb, long npts, double* part, float* gsum,
                hipStream_t s) {
  hipLaunchKernelGGL(k_loss, dim3(LOSS_BLOCKS), dim3(256), 0, s, y, tau, scale, gyb, npts, part, gsum);
  return 0;
}

// ------------------------------------------------------------------ layout conversions
__global__ void k_pack_input(const float* __restrict__ u, float scale, __bf16* __restrict__ x, long n) {
  const long p = (long)blockIdx.x * 256 + threadIdx.x;
  if (p >= n) return;
  bf16x8 v = {};
#pragma unroll
  for (int c = 0; c < 3; ++c) v[c] = (__bf16)(u[c * n + p] * scale);
  ((bf16x8*)x)[p] = v;
}
int launch_pack_input(const float* u, float scale, __bf16* x, long n, hipStream_t s) {
  hipLaunchKernelGGL(k_pack_input, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, u, scale, x, n);
  return 0;
}

// Canonical FP32 parameters -> packed bf16 layouts (one thread per packed entry).
__global__ void __launch_bounds__(256) k_pack_weights(const float* __restrict__ P, ClosureWeights w) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  // segment sizes
  constexpr int S1 = 27 * 32 * 8, S2 = 27 * 32 * 32, S3 = 27 * 16 * 32, S4 = 27 * 32 * 8, S5 = 27 * 32 * 32;
  if (i < S1) {  // w1f[tap][co][ci<8] = W1[tap][co][ci<3]
    const int ci = i % 8, co = (i / 8) % 32, tap = i / 256;
    w.w1f[i] = (__bf16)(ci < 3 ? P[CL_OW1 + (tap * 32 + co) * 3 + ci] : 0.f);
    return;
  }
  int j = i - S1;
  if (j < S2) {
    w.w2f[j] = (__bf16)P[CL_OW2 + j];
    return;
  }
  j -= S2;
  if (j < S3) {  // w3f[tap][co<16][ci] = W3[tap][co<6][ci]
    const int ci = j % 32, co = (j / 32) % 16, tap = j / 512;
    w.w3f[j] = (__bf16)(co < 6 ? P[CL_OW3 + (tap * 6 + co) * 32 + ci] : 0.f);
    return;
  }
  j -= S3;
  if (j < S4) {  // w3b[tap'][c2 (32)][c3 < 8] = W3[26 - tap'][c3 < 6][c2]
    const int c3 = j % 8, c2 = (j / 8) % 32, tp = j / 256;
    w.w3b[j] = (__bf16)(c3 < 6 ? P[CL_OW3 + ((26 - tp) * 6 + c3) * 32 + c2] : 0.f);
    return;
  }
  j -= S4;
  if (j < S5) {  // w2b[tap'][ci][co] = W2[26 - tap'][co][ci]
    const int co = j % 32, ci = (j / 32) % 32, tp = j / 1024;
    w.w2b[j] = (__bf16)P[CL_OW2 + ((26 - tp) * 32 + co) * 32 + ci];
    return;
  }
  j -= S5;
  if (j < 32) { w.b1[j] = P[CL_OB1 + j]; return; }
  j -= 32;
  if (j < 32) { w.b2[j] = P[CL_OB2 + j]; return; }
  j -= 32;
  if (j < 16) w.b3[j] = j < 6 ? P[CL_OB3 + j] : 0.f;
}
int launch_pack_weights(const float* params, const ClosureWeights& w, hipStream_t s) {
  const int n = 27 * 32 * 8 + 27 * 32 * 32 + 27 * 16 * 32 + 27 * 32 * 8 + 27 * 32 * 32 + 32 + 32 + 16;
  hipLaunchKernelGGL(k_pack_weights, dim3((n + 255) / 256), dim3(256), 0, s, params, w);
  return 0;
}

// ------------------------------------------------------------------ Adam
__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, long n, float lr, float b1, float b2, float eps, float c1, float c2) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}
int launch_adam(float* p, const float* g, float* m, float* v, long n, float lr, float b1, float b2, float eps, int t,
                hipStream_t s) {
  const float c1 = 1.f - powf(b1, (float)t), c2 = 1.f - powf(b2, (float)t);
  hipLaunchKernelGGL(k_adam, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, g, m, v, n, lr, b1, b2, eps, c1,
                     c2);
  return 0;
}

// ------------------------------------------------------------------ box filter
// One thread per coarse point; FP64 sums over the r^3 fine points.
template <typename R>
__global__ void __launch_bounds__(256) k_box_filter(const R* __restrict__ u, int N0, int N1, int N2, int r,
                                                    R* __restrict__ ub, R* __restrict__ tau) {
  const int n0 = N0 / r, n1 = N1 / r, n2 = N2 / r;
  const long nc = (long)n0 * n1 * n2, nf = (long)N0 * N1 * N2;
  const long q = (long)blockIdx.x * 256 + threadIdx.x;
  if (q >= nc) return;
  const int c2 = (int)(q % n2), c1 = (int)((q / n2) % n1), c0 = (int)(q / ((long)n2 * n1));
  double s[3] = {0, 0, 0}, ss[6] = {0, 0, 0, 0, 0, 0};
  for (int a = 0; a < r; ++a)
    for (int b = 0; b < r; ++b) {
      const long row = ((long)(c0 * r + a) * N1 + (c1 * r + b)) * N2 + (long)c2 * r;
      for (int c = 0; c < r; ++c) {
        const double x = u[row + c], y = u[nf + row + c], z = u[2 * nf + row + c];
        s[0] += x; s[1] += y; s[2] += z;
        ss[0] += x * x; ss[1] += y * y; ss[2] += z * z; ss[3] += x * y; ss[4] += x * z; ss[5] += y * z;
      }
    }
  const double inv = 1.0 / ((double)r * r * r);
  const double m0 = s[0] * inv, m1 = s[1] * inv, m2 = s[2] * inv;
  ub[q] = (R)m0; ub[nc + q] = (R)m1; ub[2 * nc + q] = (R)m2;
  tau[q] = (R)(ss[0] * inv - m0 * m0);
  tau[nc + q] = (R)(ss[1] * inv - m1 * m1);
  tau[2 * nc + q] = (R)(ss[2] * inv - m2 * m2);
  tau[3 * nc + q] = (R)(ss[3] * inv - m0 * m1);
  tau[4 * nc + q] = (R)(ss[4] * inv - m0 * m2);
  tau[5 * nc + q] = (R)(ss[5] * inv - m1 * m2);
}
int launch_box_filter(const float* u, int N0, int N1, int N2, int r, float* ubar, float* tau, hipStream_t s) {
  if (r < 1 || N0 % r || N1 % r || N2 % r) return -1;
  const long nc = (long)(N0 / r) * (N1 / r) * (N2 / r);
  hipLaunchKernelGGL((k_box_filter<float>), dim3((unsigned)((nc + 255) / 256)), dim3(256), 0, s, u, N0, N1, N2, r,
                     ubar, tau);
  return 0;
}
int launch_box_filter_f64(const double* u, int N0, int N1, int N2, int r, double* ubar, double* tau, hipStream_t s) {
  if (r < 1 || N0 % r || N1 % r || N2 % r) return -1;
  const long nc = (long)(N0 / r) * (N1 / r) * (N2 / r);
  hipLaunchKernelGGL((k_box_filter<double>), dim3((unsigned)((nc + 255) / 256)), dim3(256), 0, s, u, N0, N1, N2, r,
                     ubar, tau);
  return 0;
}

}  // namespace sdns
