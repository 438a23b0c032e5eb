// Kernel argument blocks shared by the host orchestration (sdns_abi.hip) and
// the pass kernels (sdns_kernels.hpp).  Everything is plain data passed by
// value as kernel arguments.
//
// Buffer layouts (complex elements of the working precision):
//   state  u_hat           [3][N0][N1][Nh]        Nh = N2/2+1, kz contiguous
//   W1 (x-inverse out)     [5][M0][nky][nkz]      fields u, v, w, X(kx w), X(kx v)
//   W2 (y-inverse out)     [6][M0][M1][nkz]       fields u, v, w, wx, wy, wz
//   W3 (z pass out)        [3][M0][M1][nkzo]      F_z(u x w)
//   W4 (y-forward out)     [3][M0][nkyo][nkzo]
// nky/nkz are the kept input modes of the dealiased backward transform,
// nkyo/nkzo the kept output modes of the dealiased forward transform, stored
// compactly in fftfreq order (k >= 0 first, then the negative modes).  The kz
// dimension of the work buffers is padded to nkzp / nkzop (multiples of 16
// elements) so that every row starts on a 128-byte line.
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace sdns {

// Map between FFT bins of a length-M transform and stored rows.  Kept modes
// are -neg..pos; mode k lives in bin (k mod M) and in row (k >= 0 ? k : base + k),
// where base is the stored length (N for the uncompacted state, neg+pos+1 for
// compact work buffers).
struct RowMap {
  int neg, pos, base;
};

template <typename Rt> struct P1Args {  // x-inverse of u_hat + kx products
  const void* u;      // state [3][N0][N1][Nh]
  const void* d;      // the state is u + ds d (RK stages with KEEP_RHS), or null: u
  const void* w;      // given vorticity [3][N0][N1][Nh], or null: then W1 holds
                      // the six plain x-inverses u, v, w, wx, wy, wz (no kx products)
  void* w1;           // [5][M0][Q] ([6][M0][Q] with a given vorticity)
  const void* tw;     // forward twiddles of length M0
  const Rt* kx;       // wavenumbers of axis 0 by stored index
  const Rt *ky, *kz;  // read with curl_inv only
  int curl_inv;       // with a given vorticity: the velocity is i (K/K^2) x w (u is not read)
  int N0, N1, Nh;
  RowMap x;           // kept input modes of axis 0 (base = N0)
  int y_neg, y_pos;   // kept input modes of axis 1
  int nkz, nkzp;      // kept input kz count, padded kz stride of W1
  int Q;              // nky * nkzp columns (= W1 row stride)
  Rt ds;
  int u_tiled, d_tiled, w_tiled;  // stage arrays (tile-major)
  int xb;             // W1 blocked over x
};

template <typename Rt> struct P2Args {  // y-inverse + curl assembly
  const void* w1;
  void* w2;           // [6][M0][M1][nkz]
  const void* tw;     // forward twiddles of length M1
  const Rt* ky;       // wavenumbers of axis 1 by stored index
  const Rt* kz;       // wavenumbers of axis 2
  int N1, M0;
  RowMap y;           // kept input modes of axis 1 (base = nky)
  int nkz, nkzp;
  int Q;              // M0 * nkzp
  int xb;             // W1 blocked over x
};

template <typename Rt> struct P3Args {  // z C2R x6, cross product, z R2C x3
  const void* w2;
  void* w3;           // [3][L][nkzo]
  const void* tw;     // forward twiddles of length n = M2/2
  const void* rtw;    // exp(-2 pi i p / M2), p in [0, n)
  int nkz, nkzp, nkzo, nkzop;
  int L;              // M0 * M1 lines
};

// Order of a strided pass's tiles on the XCDs (StridedArgs::run): no runs, each XCD
// one contiguous eighth.
constexpr int XCD_EIGHTHS = 30;

// Generic batched strided-axis transform: columns q = hi*cdiv + lo live at
// offset hi*hi_stride + lo; row r of a column at offset r*row_stride; field f
// (blockIdx.y) at offset f*field_stride.
template <typename Rt> struct StridedArgs {
  const void* in;
  void* out;
  const void* tw;
  int Q, cdiv, cvalid;  // column q valid if q < Q and (q mod cdiv) < cvalid
  long in_hi, in_row, in_field;
  long out_hi, out_row, out_field;
  RowMap rin, rout;
  Rt scale;           // applied to every output (1 = none)
  int run = 5;        // log2 of the tiles per run on one XCD (xcd_tile_run)
  int stream_in, stream_out;  // non-temporal loads / stores (set by the launcher
                              // when every column tile covers whole 128-byte lines)
};

// z-axis real transforms on contiguous lines: C2R (spectral lines of nk_in
// bins -> M2 reals) or R2C (M2 reals -> nk_out bins).  Field f via blockIdx.y.
template <typename Rt> struct ZArgs {
  const void* in;
  void* out;
  const void* tw;     // length n = M2/2
  const void* rtw;    // exp(-2 pi i p / M2)
  int L;
  int nk;             // spectral bins kept (input of C2R / output of R2C)
  long in_line, in_field, out_line, out_field;  // element strides
  int stream;         // R2C: non-temporal stores (set by the launcher)
  Rt scale;
};

// Layouts for the x passes, whose blocks walk a column tile through every x:
// with x slowest, each row is 0.2 to 0.6 MB from the next, and the passes ran at
// 4.0 TB/s where the y passes reach 5.3 (wider tiles did not help, data resident
// in the last-level cache did not either: address translation).
//   RK stage arrays, which only the x passes touch, are tile-major:
//     [3][tile][N0][TW], TW = 128 bytes of columns, so that a block's rows are
//     contiguous;
//   W1 (not with a given vorticity) is blocked over x: [5][M0/XB][nky][XB][nkzp].
// 256^3, before -> after: x-inverse FP64 3/2 rule 367 -> 307 us, FP32 160 -> 143;
// x-forward + RK FP64 466 -> 442; 512^3 FP32 1800 -> 1600.
template <typename Rt> constexpr int tile_w() { return 128 / (2 * (int)sizeof(Rt)); }
template <typename Rt> constexpr int tiled_cols(int Q) { return (Q + tile_w<Rt>() - 1) / tile_w<Rt>() * tile_w<Rt>(); }
constexpr int XB = 16;

enum P5Mode { P5_RHS = 0, P5_RK0 = 1, P5_RK12 = 2, P5_RK3 = 3 };

// RK4 in the P5 stages: start value u, stage right-hand sides k1..k4, stage
// states B_i = u + b_i dt k_i, sum u + sum a_i dt k_i (integrators.py:155-157).
// What the stages keep for the sum decides their traffic (F: one spectral
// field; the passes before P5 read the stage state):
//   KEEP_SUM: an accumulator that every stage reads and writes: 48 F per step,
//     21 F of it written.
//   KEEP_STATES: only the B_i; the last stage adds
//     ((B1 - u) + 2 (B2 - u) + (B3 - u)) / 3 + dt/6 k4: 39 F, 12 F written.
//   KEEP_RHS: only the k_i; whoever reads a stage state forms u + b_i dt k_i,
//     and the last stage adds the terms with the accumulator's roundings, plain
//     or compensated: 39 F, 12 F written, and 9 F more in the x-inverse pass times
//     the share of the modes that it reads (0.3 with the 2/3 rule).
// FP64 keeps the states, and so do VV and MHD in FP32 (50 steps of 32^3: 1.3e-7 and
// 1.4e-7 from FP64, with an accumulator 2.6e-7 and 2.0e-7).  FP32 NS keeps the
// accumulator's roundings: right-hand sides, except with the 3/2 rule, whose
// x-inverse reads every mode (256^3: 4.95 ms per step with the sum, 5.12 ms with
// right-hand sides).
enum RkKeep { KEEP_SUM = 0, KEEP_STATES = 1, KEEP_RHS = 2 };
template <typename Rt> constexpr int rk_keep(bool padded, bool comp) {
  return sizeof(Rt) == 8 ? KEEP_STATES : (padded && !comp ? KEEP_SUM : KEEP_RHS);
}

template <typename Rt> struct P5Args {  // x-forward + mask + pressure + diffusion + RK4 stage
  const void* w4;     // [3][M0][nkyo][nkzo]
  void* u;            // state: step base, and the result of stage 3 (P5_RHS: the input state)
  const void* s;      // stages 1..3: the stage state whose RHS this is, or the last k (KEEP_RHS)
  void* out;          // stages 0..2: the next stage state, or this stage's k (KEEP_RHS)
  void* b1;           // stage 3: B1, B2 or k1, k2; KEEP_SUM: b1 is the accumulator of all stages
  const void* b2;
  void* lo;           // compensated mode: low part of u (caller's u_lo)
  void* rhs;          // P5_RHS: rhs output; VV, P5_RK3: this stage's right-hand side (may be null)
  void* phat;         // P5_RHS: pressure output (may be null)
  const void* source; // P5_RHS: added source (may be null)
  double* partials;   // P5_RK3: per-block (energy, enstrophy) sums (may be null)
  const void* tw;     // forward twiddles of length M0
  const Rt *kx, *ky, *kz;
  int N0, N1, Nh, N2;
  RowMap x;           // kept output modes of axis 0
  int y_neg, y_pos;   // kept output modes of axis 1
  int nkzo, nkzop;    // kept output kz count, padded kz stride of W4
  int mask_nyquist;
  int st_tiled;       // s, out, b1, b2 are tile-major
  int conv_only;      // P5_RHS: write the scaled convection term only
  Rt nu, scale;
  Rt adt, bdt;        // a dt and b dt of this stage
  Rt sdt;             // KEEP_RHS: the stage state is u + sdt s
  Rt a12;             // KEEP_RHS, stage 3: a dt of stages 1 and 2 (stage 0's is adt)
  int Q;              // N1 * Nh state columns
};

// MHD in Elsasser form (solvers/MHD.py): W1 and W2 hold the six fields u, b of a
// given-vorticity pass, W3 and W4 the transforms of the nine products S00, S01,
// S02, S11, S12, S22, A01, A02, A12 (see k_mhd_z).
template <typename Rt> struct MhdZArgs {  // z C2R x6, nine products, z R2C x9
  const void* w2;
  void* w3;           // [9][L][nkzo]
  const void* tw;
  const void* rtw;
  int nkz, nkzp, nkzo, nkzop;
  int L;
};
template <typename Rt> struct MhdXArgs {  // x-forward of the products, mask, pressure, diffusion, RK4 stage
  const void* w4;     // [9][M0][nkyo][nkzo]
  // arrays of three components, [0] of U and [1] of B; roles as in P5Args with
  // KEEP_STATES (P5_RHS: u the input state, out the right-hand side); s, out of
  // stages 0..2, b1 and b2 are stage arrays, tile-major
  void* u[2];
  const void* s[2];
  void* out[2];
  const void* b1[2];
  const void* b2[2];
  void* phat;         // P5_RHS, P5_RK3: pressure output (may be null)
  void* rhs[2];       // P5_RK3: this stage's right-hand side (may be null)
  const void* tw;
  const Rt *kx, *ky, *kz;
  int N0, N1, Nh, N2;
  RowMap x;
  int y_neg, y_pos, nkzo, nkzop;
  int mask_nyquist;
  Rt visc[2];         // nu, eta
  Rt scale, adt, bdt;
  int Q;
};

// One x-plane of P2, P3 and P4 in LDS (sdns_plane.hpp).
template <typename Rt> struct PlaneArgs {
  const void* w1;
  void* w4;
  const void *twy, *twz, *rtw;  // forward twiddles of lengths M1 and M2/2, real-transform table
  const Rt *ky, *kz;
  int N1, M0;
  RowMap y, yo;       // kept input modes of axis 1 (base = nky), kept output modes (base = nkyo)
  int nkz, nkzp, nkzo, nkzop;
  int given;          // W1 holds the six fields of a given vorticity
};

// One block of a batched pass: box index (-1 for padding blocks) and the
// block's tile within that box.
struct BatchWork {
  int box, tile;
};

// LDS stride (complex elements) of one z line owned by P threads; the staged
// spectral line needs n + 1 entries.  With P >= 16 a line fills at least a
// quarter wave, and a stride of 16 modulo 32 puts the two lines of a fp32
// half-wave 32 banks apart, so their contiguous accesses share no bank.
constexpr int zslot(int n, int P) { return P >= 16 ? n + 1 + ((16 - (n + 1) % 32) + 32) % 32 : n + 1; }

// Lines per block of the LDS-assisted z scheme (three slots of stride sl per
// line within 40 KB), and the slot stride it uses: the padded stride when it
// keeps the lines per block and either the blocks that fit in a CU's 160 KB of
// LDS (twiddle tables included) or at least five of them.  Measured on the
// 256^3 z passes: padding gains 16% at n = 128 (6 -> 5 blocks per CU) and
// loses 15% at n = 192 (4 -> 3 blocks per CU).
constexpr int z3_lines(int n, int P, int esz, int sl) {
  int L = 256 / P;
  if (L < 1) L = 1;
  while (L > 1 && 3 * L * sl * esz > 40960) L /= 2;
  return L;
}
// The single-box kernel keeps the real-transform twiddles in LDS for FP32
// and reads them from global memory for FP64 (the batched kernel keeps both
// tables in LDS).
constexpr bool z3_rtw_in_lds(int esz) { return esz == 8; }
constexpr int z3_blocks_per_cu(int n, int P, int esz, int sl) {
  return 163840 / ((3 * z3_lines(n, P, esz, sl) * sl + (z3_rtw_in_lds(esz) ? 2 * n : n)) * esz);
}
constexpr int z3_slot(int n, int P, int esz) {
  return z3_lines(n, P, esz, zslot(n, P)) == z3_lines(n, P, esz, n + 1) &&
                 (z3_blocks_per_cu(n, P, esz, zslot(n, P)) >= z3_blocks_per_cu(n, P, esz, n + 1) ||
                  z3_blocks_per_cu(n, P, esz, zslot(n, P)) >= 5)
             ? zslot(n, P)
             : n + 1;
}

}  // namespace sdns
