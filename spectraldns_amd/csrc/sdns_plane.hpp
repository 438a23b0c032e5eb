// One x-plane of the convection term in LDS: y-inverse and curl assembly, z pass
// and y-forward (P2, P3 and P4 of sdns_kernels.hpp) in one kernel, for boxes whose
// six-field plane fits in a CU's LDS (y and half z lines of up to 64 and 32
// points: 68 KB at 64^3 FP32 with the 2/3 rule).
//
// W2 and W3 (12 F and 6 F of traffic per evaluation) then never reach memory, and
// three launches become one.  Single boxes of 32^3 and 64^3 are bound by launch
// and load latency (about 4 us per pass whatever its work), the ensembles of such
// boxes by the z pass's LDS work at low occupancy.
//
// Phases of a block (one plane), a block barrier between them:
//   1. y-inverse: lines (field f, kz); line f*nkz + kz lives in LDS column
//      f*nkz + kz of M1 rows of RS elements, which is also its exchange area.
//   2. z: row y holds the six spectral lines of that y.  PZ threads transform
//      them (registers, exchange in a scratch row per line), form u x w and
//      write the three spectral products over the row's own columns.
//   3. y-forward: columns i*nkzo + kz, kept rows to W4.
// All threads of a line are in one wave, so no barrier is needed inside a phase.
#pragma once
#include "sdns_kernels.hpp"

namespace sdns {

// Points per thread: as many threads per line as the block has for the plane,
// with at most two exchanges (three passes for n = 24 and 32).
constexpr int plane_EY(int M1) { return M1 == 16 ? 4 : (M1 == 24 ? 6 : (M1 == 48 ? 12 : 8)); }
constexpr int plane_EZ(int n) { return n == 24 ? 6 : (n == 12 ? 6 : 4); }
// Row stride: odd, so that the rows of a column fall on different banks.
__host__ __device__ constexpr int plane_rs(int nkz) { return 6 * nkz + 1; }
template <int M1, int n, int TH> struct PlaneCfg {
  static constexpr int EY = plane_EY(M1), PY = M1 / EY, EZ = plane_EZ(n), PZ = n / EZ;
  static constexpr int LZ = TH / PZ < M1 ? TH / PZ : M1;  // z lines per round
  static_assert(64 % PY == 0 && 64 % PZ == 0, "a line's threads share one wave");
};
// LDS bytes: plane, z scratch, twiddle tables.
template <int M1, int n, int TH> constexpr size_t plane_lds(int nkz, int esz) {
  return (size_t)(M1 * plane_rs(nkz) + PlaneCfg<M1, n, TH>::LZ * (n + 1) + M1 + 2 * n) * esz;
}

// Z[t + P e] of a spectral row of nk <= NKI bins: own bins and partners that lie
// at or above NKI for every thread are compile-time zeros.
template <typename Rt, int n, int E, int NKI>
__device__ __forceinline__ void plane_c2r(cx<Rt> (&z)[E], const cx<Rt>* my, int nk, const cx<Rt>* rtw, int t) {
  using C = cx<Rt>;
  constexpr int P = n / E;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int p = t + P * e;
    C xa = czero<C>(), xb = czero<C>();
    if (P * e < NKI) xa = p < nk ? my[p] : czero<C>();
    if (n - (P * e + P - 1) < NKI) xb = n - p < nk ? my[n - p] : czero<C>();
    if (e == 0 && p == 0) { xa.y = 0; xb.y = 0; }
    const C ev = mk<C>(xa.x + xb.x, xa.y - xb.y);
    const C d = mk<C>(xa.x - xb.x, xa.y + xb.y);
    const C od = cmulc(d, rtw[p]);
    z[e] = mk<C>(ev.x - od.y, ev.y + od.x);
  }
}

// NKI: bound of the kept input bins (2/3 and 3/2 rule), or n + 1.
template <typename Rt, int M1, int n, int TH, int NKI>
__device__ __forceinline__ void plane_body(const PlaneArgs<Rt>& a, int x, cx<Rt>* sm) {
  using C = cx<Rt>;
  using Cfg = PlaneCfg<M1, n, TH>;
  constexpr int EY = Cfg::EY, PY = Cfg::PY, CY = 64 / PY, EZ = Cfg::EZ, PZ = Cfg::PZ, LZ = Cfg::LZ;
  const int nkz = a.nkz, nkzo = a.nkzo, RS = plane_rs(nkz);
  C* pl = sm;
  C* scr = pl + M1 * RS;
  C* twy = scr + LZ * (n + 1);
  C* twz = twy + M1;
  C* rtw = twz + n;
  for (int i = threadIdx.x; i < M1; i += TH) twy[i] = ((const C*)a.twy)[i];
  for (int i = threadIdx.x; i < n; i += TH) {
    twz[i] = ((const C*)a.twz)[i];
    rtw[i] = ((const C*)a.rtw)[i];
  }
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int cy = lane % CY, ty = lane / CY;  // y lines: CY columns x PY threads per wave
  constexpr int NW = TH / 64;
  // ---- y-inverse and curl assembly (p2_body): u, v, w, wx, wy, wz
  {
    using F = LineFFT<Rt, M1, EY, +1, true>;
    const long wfield = (long)a.M0 * a.y.base * a.nkzp;
    const C* __restrict__ w1 = (const C*)a.w1 + (long)x * a.y.base * a.nkzp;
    const int nl = 6 * nkz;
    bool first = true;
    for (int c0 = wave * CY; c0 < nl; c0 += NW * CY) {
      const int li = c0 + cy;
      const bool valid = li < nl;
      const int f = valid ? li / nkz : 0, kz = valid ? li - f * nkz : 0;
      // wx = i(ky W - kz V), wy = i(kz U - X(kx W)), wz = i(X(kx V) - ky U)
      const bool curl = f >= 3 && !a.given;
      const int fa = !curl ? f : (f == 3 ? 2 : (f == 4 ? 0 : 4)), fb = f == 3 ? 1 : (f == 4 ? 3 : 0);
      const Rt kzv = a.kz[kz];
      C v[EY], b[EY];
#pragma unroll
      for (int e = 0; e < EY; ++e) {
        const int r = valid ? bin_row(ty + PY * e, M1, a.y) : -1;
        v[e] = r >= 0 ? w1[fa * wfield + (long)r * a.nkzp + kz] : czero<C>();
        b[e] = r >= 0 && curl ? w1[fb * wfield + (long)r * a.nkzp + kz] : czero<C>();
      }
      if (curl) {
#pragma unroll
        for (int e = 0; e < EY; ++e) {
          const int p = ty + PY * e;
          const int k = p <= a.y.pos ? p : p - M1;
          const Rt ky = bin_row(p, M1, a.y) >= 0 ? a.ky[k >= 0 ? k : a.N1 + k] : Rt(0);
          const Rt ca = f == 3 ? ky : (f == 4 ? kzv : Rt(1)), cb = f == 3 ? kzv : (f == 4 ? Rt(1) : ky);
          v[e] = cmuli<1>(mk<C>(ca * v[e].x - cb * b[e].x, ca * v[e].y - cb * b[e].y));
        }
      }
      if (first) __syncthreads();  // twiddle tables (every wave runs the first round)
      first = false;
      C* col = pl + (valid ? li : 0);
      if (valid) {
        F::run(v, ty, col, RS, twy);
#pragma unroll
        for (int e = 0; e < EY; ++e) col[(ty + PY * e) * RS] = v[e];
      }
    }
    if (first) __syncthreads();
  }
  __syncthreads();
  // ---- z: C2R of six fields, u x w, R2C of three
  {
    using Fi = LineFFT<Rt, n, EZ, +1, true>;
    using Ff = LineFFT<Rt, n, EZ, -1, true>;
    const int t = threadIdx.x % PZ, l = threadIdx.x / PZ;
    C* my = scr + (l < LZ ? l : 0) * (n + 1);
    if (l < LZ) {
      for (int y = l; y < M1; y += LZ) {
        C* row = pl + y * RS;
        C g[6][EZ];
#pragma unroll
        for (int f = 0; f < 6; ++f) {
          plane_c2r<Rt, n, EZ, NKI>(g[f], row + f * nkz, nkz, rtw, t);
          Fi::run(g[f], t, my, 1, twz);
        }
        lds_barrier<true>();
#pragma unroll
        for (int e = 0; e < EZ; ++e) {
          const C u0 = g[0][e], u1 = g[1][e], u2 = g[2][e];
          const C w0 = g[3][e], w1 = g[4][e], w2 = g[5][e];
          g[0][e] = mk<C>(u1.x * w2.x - u2.x * w1.x, u1.y * w2.y - u2.y * w1.y);
          g[1][e] = mk<C>(u2.x * w0.x - u0.x * w2.x, u2.y * w0.y - u0.y * w2.y);
          g[2][e] = mk<C>(u0.x * w1.x - u1.x * w0.x, u0.y * w1.y - u1.y * w0.y);
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          Ff::run(g[i], t, my, 1, twz);
#pragma unroll
          for (int e = 0; e < EZ; ++e) my[t + PZ * e] = g[i][e];
          lds_barrier<true>();
          C* out = row + i * nkzo;
#pragma unroll
          for (int e = 0; e < EZ; ++e) {
            const int k = t + PZ * e;
            const C X = r2c_bin(g[i][e], my[(n - k) % n], rtw[k]);
            if (k < nkzo) out[k] = X;
            if (k == 0 && nkzo > n) out[n] = mk<C>(g[i][e].x - g[i][e].y, Rt(0));
          }
          lds_barrier<true>();
        }
      }
    }
  }
  __syncthreads();
  // ---- y-forward
  {
    using F = LineFFT<Rt, M1, EY, -1, true>;
    const long wfield = (long)a.M0 * a.yo.base * a.nkzop;
    C* __restrict__ w4 = (C*)a.w4 + (long)x * a.yo.base * a.nkzop;
    const int nl = 3 * nkzo;
    for (int c0 = wave * CY; c0 < nl; c0 += NW * CY) {
      const int li = c0 + cy;
      if (li >= nl) continue;
      const int i = li / nkzo, kz = li - i * nkzo;
      C* col = pl + li;
      C v[EY];
#pragma unroll
      for (int e = 0; e < EY; ++e) v[e] = col[(ty + PY * e) * RS];
      lds_barrier<true>();
      F::run(v, ty, col, RS, twy);
#pragma unroll
      for (int e = 0; e < EY; ++e) {
        const int r = bin_row(ty + PY * e, M1, a.yo);
        if (r >= 0) st_stream(w4 + (i * wfield + (long)r * a.nkzop + kz), v[e]);
      }
    }
  }
}

// Input bins of the dealiased rules: ceil(2n/3) with the 2/3 rule, 2n/3 with the
// 3/2 rule.
constexpr int plane_nki(int n) { return (2 * n + 2) / 3; }
template <typename Rt, int M1, int n, int TH, bool RULE>
__global__ void __launch_bounds__(TH, 2) k_plane(PlaneArgs<Rt> a) {
  extern __shared__ __align__(16) unsigned char plane_smem[];
  plane_body<Rt, M1, n, TH, (RULE ? plane_nki(n) : n + 1)>(a, blockIdx.x, (cx<Rt>*)plane_smem);
}
// Batched: work items (box, plane) of the boxes with these line lengths.
template <typename Rt, int M1, int n, int TH, bool RULE>
__global__ void __launch_bounds__(TH, 2) k_batch_plane(const PlaneArgs<Rt>* __restrict__ args,
                                                       const BatchWork* __restrict__ work) {
  extern __shared__ __align__(16) unsigned char plane_smem[];
  const BatchWork w = work[blockIdx.x];
  if (w.box < 0) return;
  const PlaneArgs<Rt> a = args[w.box];
  plane_body<Rt, M1, n, TH, (RULE ? plane_nki(n) : n + 1)>(a, w.tile, (cx<Rt>*)plane_smem);
}

// ------------------------------------------------------------------ launchers
// Compiled pairs (y length, half z length): every pair of the small sides, and
// the padded 24 x 24 plane.  Block sizes of a single box: 512 threads from 48 rows
// on (a box has few planes, so the threads are what fills a CU), except the FP64
// 64-row plane, whose LDS leaves room for 32 scratch rows; the ensembles' blocks
// are 256 threads, so that two of the largest share a CU.
#define SDNS_PLANE_PAIRS(X)                                                                       \
  X(16, 8) X(16, 16) X(16, 24) X(16, 32) X(32, 8) X(32, 16) X(32, 24) X(32, 32) X(24, 12)         \
  X(48, 8) X(48, 16) X(48, 24) X(48, 32) X(64, 8) X(64, 16) X(64, 24) X(64, 32)
constexpr int plane_threads(int M1, int esz) { return M1 < 48 || (M1 == 64 && esz == 16) ? 256 : 512; }
constexpr size_t PLANE_LDS_MAX = 163840;

template <typename F> int plane_dispatch(int M1, int n, F go) {
#define SDNS_X(m, h) \
  if (M1 == m && n == h) return go(std::integral_constant<int, m>{}, std::integral_constant<int, h>{});
  SDNS_PLANE_PAIRS(SDNS_X)
#undef SDNS_X
  return -1;
}
template <typename K> int plane_allow(K kernel, size_t bytes) {
  // dynamic LDS beyond 64 KB must be allowed for the kernel (on the current device)
  return bytes > 65536 && hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess
             ? -1
             : 0;
}
template <typename Rt> int launch_plane(int M1, int n, const PlaneArgs<Rt>& a, hipStream_t s) {
  return plane_dispatch(M1, n, [&](auto mm, auto nn) {
    constexpr int m = decltype(mm)::value, h = decltype(nn)::value, TH = plane_threads(m, (int)sizeof(cx<Rt>));
    const size_t bytes = plane_lds<m, h, TH>(a.nkz, (int)sizeof(cx<Rt>));
    if (bytes > PLANE_LDS_MAX) return -1;
    const auto k = a.nkz <= plane_nki(h) ? &k_plane<Rt, m, h, TH, true> : &k_plane<Rt, m, h, TH, false>;
    if (plane_allow(k, bytes)) return -1;
    hipLaunchKernelGGL(k, dim3(a.M0), dim3(TH), bytes, s, a);
    return 0;
  });
}
// Whether a box of M0 planes runs launch_plane (its plan lays out the work buffers
// for it): where the plane fits in LDS, except few planes of the largest sizes,
// whose few blocks leave the chip idle longer than three launches take.  Per
// evaluation, three passes against the plane launch, with M0 = M1: FP32 32^2 18
// against 10 us, 48^2 24 against 15, 64^2 16 against 19; FP64 21 against 11, 30
// against 19, 22 against 34; the plane launch's time stays the same up to 256
// planes (FP64 64^2: 38 us at 256).  Steps of 8 to 512 planes of every compiled
// pair, both precisions, with the 2/3 rule and without (496 boxes): the plane
// launch takes 0.48 to 1.0 of the three passes' step, but for FP64 planes of 32 or
// 48 rows with 64-point z lines: 8 planes 116 against 108 us (32 rows) and 131
// against 117 (48), 32 planes 125 against 122 and 143 against 138, even from 48 on.
template <typename Rt> bool plane_fits(int M0, int M1, int n, int nkz) {
  if (M1 == 64 && n == 32 && M0 < (sizeof(Rt) == 4 ? 128 : 192)) return false;
  if (sizeof(Rt) == 8 && M1 >= 32 && n == 32 && M0 < 48) return false;
  return plane_dispatch(M1, n, [&](auto mm, auto nn) {
           constexpr int m = decltype(mm)::value, h = decltype(nn)::value, TH = plane_threads(m, (int)sizeof(cx<Rt>));
           return plane_lds<m, h, TH>(nkz, (int)sizeof(cx<Rt>)) <= PLANE_LDS_MAX ? 0 : -1;
         }) == 0;
}
// Batched: cubic planes (M1 = 2 n) only.
template <typename Rt> bool batch_plane_fits(int M1, int n, int nkz) {
  if (M1 != 2 * n) return false;
  return plane_dispatch(M1, n, [&](auto mm, auto nn) {
           constexpr int m = decltype(mm)::value, h = decltype(nn)::value;
           return plane_lds<m, h, 256>(nkz, (int)sizeof(cx<Rt>)) <= PLANE_LDS_MAX ? 0 : -1;
         }) == 0;
}
template <typename Rt> int launch_batch_plane(int M1, int nkz, const PlaneArgs<Rt>* args, const BatchWork* work,
                                              int nwork, hipStream_t s) {
  return plane_dispatch(M1, M1 / 2, [&](auto mm, auto nn) {
    constexpr int m = decltype(mm)::value, h = decltype(nn)::value;
    if constexpr (m != 2 * h) {
      return -1;
    } else {
      const size_t bytes = plane_lds<m, h, 256>(nkz, (int)sizeof(cx<Rt>));
      const auto k = nkz <= plane_nki(h) ? &k_batch_plane<Rt, m, h, 256, true> : &k_batch_plane<Rt, m, h, 256, false>;
      if (plane_allow(k, bytes)) return -1;
      hipLaunchKernelGGL(k, dim3(nwork), dim3(256), bytes, s, args, work);
      return 0;
    }
  });
}

}  // namespace sdns

#define SDNS_PLANE_INSTANTIATE(Rt)                                                                              \
  namespace sdns {                                                                                              \
  template int launch_plane<Rt>(int, int, const PlaneArgs<Rt>&, hipStream_t);                                   \
  template bool plane_fits<Rt>(int, int, int, int);                                                             \
  template bool batch_plane_fits<Rt>(int, int, int);                                                            \
  template int launch_batch_plane<Rt>(int, int, const PlaneArgs<Rt>*, const BatchWork*, int, hipStream_t);      \
  }
