// Single-system dense LU with partial pivoting for any order (n <= 32768), its solves, the
// determinant and the inverse from the factors.
//
// Replaces, for one system of any size:
//   solve(A, x, b) / solve(A, X, B)  (blaze/math/dense/LSE.h:6343-6373 -> solveNxN, LSE.h:5229-5257
//     -> gesv -> dgesv_, blaze/math/lapack/clapack/gesv.h:207)       -> bzg_dgesv
//   getrf (blaze/math/lapack/clapack/getrf.h:190-197), lu() (blaze/math/dense/LU.h:98-140)
//                                                                     -> bzg_dgetrf
//   getrs (blaze/math/lapack/clapack/getrs.h:207-215)                 -> bzg_dgetrs
//   det() for N > 6 (blaze/math/expressions/DMatDetExpr.h:324-357)    -> bzg_ddet_lu
//   invert()/inv() by LU (blaze/math/dense/Inversion.h:3337-3347)     -> bzg_dgetri
// The batched kernels (lu.hip) keep serving orders <= 512 with <= 8 right-hand sides.
//
// Matrices are row-major (the math matrix A, leading dimension lda); P A = L U with L unit
// lower, U upper, ipiv 1-based (row i was interchanged with row ipiv[i] - 1, in order) and
// info the 1-based column of the first exactly-zero pivot: the results of LAPACK dgetrf on A.
//
// Factorisation: panels of 64 columns, each followed by its interchanges and U12 = L11^-1 A12 on every
// other column (panel_swap_kernel) and A22 -= L21 U12 through bzg_dgemm on the FP64 matrix cores;
// blocks wider than 2048 columns are split in half first (dgetrf2's recursion), so that their
// updates have more work per byte.  A panel is factored in leaves of up to 16 columns, each held in the
// registers of one workgroup (getf2_leaf_kernel), with a rank-16 update of the panel's remaining columns
// over the device (rank_update_kernel) in between.  Solves with few right-hand sides take one launch
// per 64 rows and direction (trsv_block_kernel), others recurse on 64-row blocks and bzg_dgemm.
// n = 3000 with 16 right-hand sides: 12.6 ms; 28.1 ms with leaves of 8 columns and dgetrf2's recursion
// down to them (708 triangular solves of 32 rows, 796 small products).  n = 8192: 55 ms (99 ms), 16384 349
// (420), 25000 928 (1168): above 8192 rows a leaf holds two columns, above 16384 one, and those
// instances spill (48 and 20 registers a lane).
#include "common.hpp"

#include <cfloat>
#include <climits>
#include <algorithm>
#include <mutex>

namespace bzg {
namespace big {

constexpr int kPanel = 64;      // columns of a panel
constexpr int kTrsmLeaf = 32;
constexpr int64_t kMaxOrder = 32768;

// Original position of what ends at position `pos` after the interchanges base + j <-> piv[j]
// (j = 0 .. w - 1, in order): the interchanges followed backwards.
__device__ __forceinline__ int swap_source(int pos, const int* piv, int base, int w) {
#pragma unroll 8
  for (int j = w - 1; j >= 0; --j) {
    const int pj = piv[j];
    if (pos == base + j) pos = pj;
    else if (pos == pj) pos = base + j;
  }
  return pos;
}

// ---- leaf of a panel: columns c0 .. c0 + w - 1 (w <= WL) on rows c0 .. n - 1 ------------------
// The panel is the columns p0 .. p0 + nbp - 1 (nbp <= 64).  Thread t of T holds the block's rows
// t + T i, i < R (m = n - c0 <= T R).
//
// Bound by latency: a column is one chain of some 350 dependent instructions on one workgroup,
// about 1.3 us.  Per column: a per-thread maximum over R rows, an integer DPP maximum of the high
// words over the wavefront, a barrier, the best of the wavefronts, the chosen row to LDS, a
// barrier, and the rank-1 update in registers.  Sixteen columns at 500 rows take 27 us in all (load,
// store and the other columns included), 12 at 3000 rows 36 us; eight took 21 and 35 us with
// shuffled (value, row) pairs, rows moved between registers and one leaf per 8 columns.
//   * Rows never move between registers.  The row chosen at step j stays in LDS as row j of the
//     result; its register copy becomes NaN, which no maximum picks again.  The row at position j
//     takes the chosen row's position; only the first w rows (slot 0 of threads 0 .. w - 1) are
//     ever displaced, so one register holds a thread's position.
//   * The registers rotate by one column a step (at step j, a[i][c] is column (c + j) % WL, the
//     finished columns last), so the loop stays rolled with constant register indices: expanded,
//     its code runs from memory once per launch and the instruction fetches cost 2 to 4 us a column.
//   * Rows past the matrix are NaN: no candidates without a mask, and never stored.
//   * One lane's LDS access occupies the LDS for as long as a full wavefront's: only the chosen row
//     is written, after the choice, by one wavefront.
// The leaf also applies its interchanges to the panel's other columns and forms U12 = L11^-1 A12
// for those on its right (the rows it needs are fetched as they are chosen), so a panel needs one
// more launch per leaf (rank_update_kernel) only.
struct LeafBest {
  double v;       // a wavefront's largest |a| (-1: none)
  int pos, phys;  // that row's position and place (thread + T slot)
};
template <int T, int WL>
struct LeafShm {
  LeafBest best[2][T / 64];  // by step parity
  LeafBest diag[2];          // the row at position j: its value, thread
  double row[WL][WL];        // the rows chosen, each in its step's column order
  int piv[WL], phys[WL];     // positions and places chosen
  double l11[WL][WL + 2];
  double top[WL][kPanel];  // the block's rows of the panel's other columns
  int dst[WL];             // first w rows: final position, -1 when chosen
};

template <int T, int R, int WL>
__global__ __launch_bounds__(T) void getf2_leaf_kernel(double* __restrict__ A, long lda, int n, int c0, int w, int p0,
                                                       int nbp, int32_t* __restrict__ ipiv,
                                                       int32_t* __restrict__ info) {
  constexpr int NW = T / 64;
  constexpr int NQ = (WL + NW - 1) / NW;  // rows of the block per wavefront
  static_assert(NW == 8 || NW == 4, "four or eight wavefronts");
  __shared__ LeafShm<T, WL> sh;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int m = n - c0;
  double* P = A + (long)c0 * lda + c0;
  const double nan = __builtin_nan("");
  // a full-width row of 4, 8, 12 or 16 columns moves as 32-byte vectors (fewer load instructions:
  // what limits one workgroup's share of the memory bandwidth), others element by element
  double a[R][WL];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int row = t + T * i;
    if (WL % 4 == 0 && w == WL) {
#pragma unroll
      for (int c4 = 0; c4 < WL / 4; ++c4) {
        dvec4u v = {nan, nan, nan, nan};
        if (row < m) v = *reinterpret_cast<const dvec4u*>(P + (long)row * lda + 4 * c4);
        a[i][4 * c4] = v[0]; a[i][4 * c4 + 1] = v[1]; a[i][4 * c4 + 2] = v[2]; a[i][4 * c4 + 3] = v[3];
      }
    } else {
#pragma unroll
      for (int c = 0; c < WL; ++c) a[i][c] = (row < m && c < w) ? P[(long)row * lda + c] : nan;
    }
  }
  // the panel's other columns, one per lane: wavefront q % NW fetches the block's row q now and the
  // row chosen at step q after the last step
  const bool other = lane < nbp - w;
  const int col = p0 + (lane < c0 - p0 ? lane : lane + w);
  double own[NQ], got[NQ];
#pragma unroll
  for (int u = 0; u < NQ; ++u) {
    const int q = wave + NW * u;
    own[u] = (other && q < w) ? A[(long)(c0 + q) * lda + col] : 0.0;
  }
  int pos0 = t;       // position of the row in slot 0
  unsigned long long used = 0;  // slots whose row was chosen
  int first_zero = 0;
#pragma unroll 1
  for (int j = 0; j < WL; ++j) {
    double pv[WL];
    const bool step = j < w;
    if (step) {
      const int par = j & 1;
      // the thread's largest |a| and its slot (positions grow with the slot, but for a displaced
      // slot 0, which loses a tie to a lower position)
      double bv = a[0][0] == a[0][0] ? fabs(a[0][0]) : -1.0;
      int bs = 0;
#pragma unroll
      for (int i = 1; i < R; ++i) {
        const bool g = fabs(a[i][0]) > bv;
        bv = g ? fabs(a[i][0]) : bv;
        bs = g ? i : bs;
      }
      if (t < w && pos0 != t && bs == 0) {
#pragma unroll
        for (int i = R - 1; i >= 1; --i)
          if (fabs(a[i][0]) == bv && t + T * i < pos0) bs = i;
      }
      const int bp = bs == 0 ? pos0 : t + T * bs;
      // the wavefront's best: lane 63 ends with the largest high word
      int k = high_word(bv);
      k = max(k, dpp<0x111>(k));  // row_shr:1
      k = max(k, dpp<0x112>(k));  // row_shr:2
      k = max(k, dpp<0x114>(k));  // row_shr:4
      k = max(k, dpp<0x118>(k));  // row_shr:8
      k = max(k, dpp<0x142>(k));  // row_bcast:15
      k = max(k, dpp<0x143>(k));  // row_bcast:31
      k = __builtin_amdgcn_readlane(k, 63);
      const int src = k < 0 ? 0 : best_lane(__ballot(high_word(bv) == k), bv, bp);
      if (lane == src) sh.best[par][wave] = LeafBest{bv, bp, t + T * bs};
      if (t < w && pos0 == j) sh.diag[par] = LeafBest{a[0][0], j, t};  // one of the first w rows
      __syncthreads();
      const LeafBest c = sh.best[par][lane & (NW - 1)];
      const LeafBest d = sh.diag[par];
      k = high_word(c.v);
      k = max(k, dpp<0xb1>(k));                  // lanes ^ 1
      k = max(k, dpp<0x4e>(k));                  // lanes ^ 2
      if (NW == 8) k = max(k, dpp<0x141>(k));  // mirrored in 8
      const int gw = best_lane(__ballot(high_word(c.v) == k) & ((1ull << NW) - 1), c.v, c.pos);
      int gr = __builtin_amdgcn_readlane(c.pos, gw);
      int phys = __builtin_amdgcn_readlane(c.phys, gw);
      if (__builtin_amdgcn_readfirstlane((int)(d.v != d.v))) {  // idamax keeps a NaN at position j
        gr = j;
        phys = __builtin_amdgcn_readfirstlane(d.phys);
      }
      // the chosen row: its values to LDS, out of the candidates; the row at position j takes its
      // position
      const int ip = phys / T;
      if (wave == phys % T / 64 && t == phys % T) {
        used |= 1ull << ip;
#pragma unroll
        for (int i = 0; i < R; ++i)
          if (i == ip) {
#pragma unroll
            for (int q = 0; q < WL; ++q) sh.row[j][q] = a[i][q];
            a[i][0] = nan;
          }
        if (ip == 0) pos0 = INT_MAX;
        sh.piv[j] = c0 + gr;
        sh.phys[j] = phys;
      }
      if (pos0 == j && t < w) pos0 = gr;
      double rinv = 1.0 / lane_value(c.v, gw);
      __asm__ volatile("" : "+v"(rinv));  // before the barrier, while the row is written
      __syncthreads();
#pragma unroll
      for (int q = 0; q < WL; ++q) pv[q] = sh.row[j][q];
      const double piv = pv[0];
      rinv = piv < 0.0 ? -rinv : rinv;
      if (piv != piv) rinv = piv;
      const bool nz = __builtin_amdgcn_readfirstlane((int)(piv != 0.0)) != 0;
      const bool tiny = __builtin_amdgcn_readfirstlane((int)(fabs(piv) < DBL_MIN)) != 0;
      // scale by the reciprocal (divide when |pivot| < DBL_MIN, dgetf2's sfmin rule; nothing for a
      // zero pivot)
      if (nz && !tiny) {
#pragma unroll
        for (int i = 0; i < R; ++i) a[i][0] *= rinv;
      } else if (nz) {
#pragma unroll
        for (int i = 0; i < R; ++i) a[i][0] /= piv;
      }
      if (!nz && first_zero == 0) first_zero = c0 + j + 1;
    }
    // the rank-1 update of the WL - 1 - j columns to the right (applied for a zero pivot too, as
    // dger is), every column moving one register down; the finished ones only move
    double l[R];
#pragma unroll
    for (int i = 0; i < R; ++i) l[i] = a[i][0];
#pragma unroll
    for (int c = 1; c < WL; ++c) {
      if (step && c < WL - j) {
        __asm__ volatile("");  // a branch, not an update and a selection
#pragma unroll
        for (int i = 0; i < R; ++i) a[i][c - 1] = a[i][c] - l[i] * pv[c];
      } else {
#pragma unroll
        for (int i = 0; i < R; ++i) a[i][c - 1] = a[i][c];
      }
    }
#pragma unroll
    for (int i = 0; i < R; ++i) a[i][WL - 1] = l[i];
  }
#pragma unroll
  for (int u = 0; u < NQ; ++u) {
    const int q = wave + NW * u;
    const int phys = __builtin_amdgcn_readfirstlane(q < w ? sh.phys[q] : 0);
    got[u] = (other && q < w) ? A[(long)(c0 + phys) * lda + col] : 0.0;
  }
  // the rows fetched from the other columns have arrived before any row is overwritten
  if (t < w) sh.dst[t] = (used & 1ull) ? -1 : pos0;
#pragma unroll
  for (int u = 0; u < NQ; ++u) {
    const int q = wave + NW * u;
    if (q < WL) sh.top[q][lane] = got[u];
  }
  __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  // the chosen rows: the block's first w rows
  for (int e = t; e < w * WL; e += T) {
    const int j = e / WL, c = e % WL;
    const double x = sh.row[j][c >= j ? c - j : c - j + WL];
    sh.l11[j][c] = x;
    if (c < w) P[(long)j * lda + c] = x;
  }
  if (t < w) ipiv[c0 + t] = sh.piv[t] + 1;
  if (t == 0 && first_zero && *info == 0) *info = first_zero;
  // the other columns' displaced rows
#pragma unroll
  for (int u = 0; u < NQ; ++u) {
    const int q = wave + NW * u;
    if (q < w) {
      const int d = __builtin_amdgcn_readfirstlane(sh.dst[q]);
      if (other && d >= 0) A[(long)(c0 + d) * lda + col] = own[u];
    }
  }
  __syncthreads();  // l11
  // the remaining rows, at their final positions
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int row = t + T * i;
    const int to = i == 0 ? pos0 : row;
    if (row < m && !(used >> i & 1ull)) {
      if (WL % 4 == 0 && w == WL) {
#pragma unroll
        for (int c4 = 0; c4 < WL / 4; ++c4)
          *reinterpret_cast<dvec4u*>(P + (long)to * lda + 4 * c4) =
              dvec4u{a[i][4 * c4], a[i][4 * c4 + 1], a[i][4 * c4 + 2], a[i][4 * c4 + 3]};
      } else {
#pragma unroll
        for (int c = 0; c < WL; ++c)
          if (c < w) P[(long)to * lda + c] = a[i][c];
      }
    }
  }
  if (wave == 0 && other) {  // U12, while the stores drain
    double x[WL];
#pragma unroll
    for (int i = 0; i < WL; ++i) x[i] = sh.top[i][lane];
    if (col >= c0 + w) {
#pragma unroll
      for (int i = 1; i < WL; ++i)
        if (i < w) {
#pragma unroll
          for (int k = 0; k < i; ++k) x[i] -= x[k] * sh.l11[i][k];
        }
    }
#pragma unroll
    for (int i = 0; i < WL; ++i)
      if (i < w) A[(long)(c0 + i) * lda + col] = x[i];
  }
}

// A22 -= L21 U12 inside a panel: rows r0 .. n - 1, columns r0 .. r0 + nc - 1 (nc <= 64) with the WL
// columns of L21 and rows of U12 just before r0.  A lane holds one column of U12; the rows of L21
// are uniform over the wavefront (scalar loads).  A few microseconds of latency: 4 rows a
// wavefront spread the rows over the device.
constexpr int kRankRows = 4;
template <int WL>
__global__ __launch_bounds__(256) void rank_update_kernel(double* __restrict__ A, const double* __restrict__ L,
                                                          const double* __restrict__ U, long lda, int n, int r0,
                                                          int nc) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row0 = r0 + (blockIdx.x * 4 + wave) * kRankRows;
  if (row0 >= n) return;
  const int nr = min(kRankRows, n - row0);
  const int lc = min(lane, nc - 1);
  double u[WL], x[kRankRows];
#pragma unroll
  for (int k = 0; k < WL; ++k) u[k] = U[(long)(r0 - WL + k) * lda + r0 + lc];
#pragma unroll
  for (int i = 0; i < kRankRows; ++i) x[i] = A[(long)(row0 + min(i, nr - 1)) * lda + r0 + lc];
#pragma unroll
  for (int i = 0; i < kRankRows; ++i) {
    const double* l = L + (long)(row0 + min(i, nr - 1)) * lda + r0 - WL;
#pragma unroll
    for (int k = 0; k < WL; ++k) x[i] -= l[k] * u[k];
  }
#pragma unroll
  for (int i = 0; i < kRankRows; ++i)
    if (i < nr && lane < nc) A[(long)(row0 + i) * lda + r0 + lane] = x[i];
}

// ---- 64-row triangular solves on LDS tiles ------------------------------------------------------
// A 64 x 64 diagonal block of factors (padded to the identity), the reciprocals of its diagonal and,
// per wavefront that loaded it, whether it holds an infinity or a NaN.
struct Diag64 {
  double l[kPanel][kPanel + 2];  // row stride 66: the MFMA operand reads hit 64 different banks
  double rinv[kPanel];
  int special[4];
};

template <bool UPPER>
__device__ __forceinline__ void load_diag64(Diag64& d, const double* __restrict__ T, long ldt, int nb) {
  const int c = threadIdx.x & 63, w = threadIdx.x >> 6;
  double v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int r = w + 4 * i;
    v[i] = (r < nb && c < nb) ? T[(long)r * ldt + c] : (r == c ? 1.0 : 0.0);
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int r = w + 4 * i;
    d.l[r][c] = v[i];
    if (UPPER && r == c) d.rinv[r] = 1.0 / v[i];
  }
  int top = 0;  // the largest exponent field
#pragma unroll
  for (int i = 0; i < 16; ++i) top = max(top, high_word(v[i]) & 0x7ff00000);
  top = __any(top == 0x7ff00000);
  if (c == 0) d.special[w] = top;
}

__device__ __forceinline__ bool has_special(const Diag64& d) {
  return __builtin_amdgcn_readfirstlane(d.special[0] | d.special[1] | d.special[2] | d.special[3]) != 0;
}

// x / d from r = 1 / d, which is off the column's chain: the product and one correction by its remainder
// (P. Markstein, "Computation of elementary functions on the IBM RISC System/6000 processor", IBM J.
// Res. Dev. 34, 1990: with r correctly rounded and the product within an ulp, the corrected quotient is
// the rounded one); the division itself where the product or its remainder may leave the range of
// normal numbers.
__device__ __forceinline__ double divide_by(double x, double d, double r) {
  double q = x * r;
  q = fma(fma(-q, d, x), r, q);
  if (!(fabs(q) > 1e-280 && fabs(q) < 1e280 && fabs(r) > 1e-300 && fabs(r) < 1e300 && fabs(x) > 1e-250)) q = x / d;
  return q;
}

// Part s (rows 16 s .. 16 s + 15) of T x = b for one column in x[], by substitution in the order of
// reference dtrsm (Left, NoTrans): for each k, skip a zero x(k), scale by the diagonal (upper),
// subtract x(k) T(i, k).
template <bool UPPER>
__device__ __forceinline__ void substitute16(double (&x)[16], const Diag64& d, int s) {
#pragma unroll
  for (int k0 = 0; k0 < 16; ++k0) {
    const int k = UPPER ? 15 - k0 : k0;
    if (x[k] != 0.0) {
      if (UPPER) x[k] = divide_by(x[k], d.l[16 * s + k][16 * s + k], d.rinv[16 * s + k]);
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (UPPER ? i < k : i > k) x[i] -= x[k] * d.l[16 * s + i][16 * s + k];
    }
  }
}

// Rows 16 q .. 16 q + 15 of X minus T's columns 16 s .. 16 s + 15 times the solved part s, by one
// wavefront.  FP64 MFMAs multiply a zero x(k) like any other; where the block holds an infinity or a NaN
// that would make a NaN of a row that substitution never touches, so there the zeros are skipped.
__device__ __forceinline__ void subtract_part16(double (*X)[16], const Diag64& d, int q, int s, bool special, int lane) {
  const int r16 = lane & 15, g = lane >> 4;
  d4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = X[16 * q + 4 * i + g][r16];
  if (__builtin_expect(special, 0)) {
#pragma unroll 1
    for (int k = 0; k < 16; ++k) {
      const double x = X[16 * s + k][r16];
      if (x != 0.0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] -= x * d.l[16 * q + 4 * i + g][16 * s + k];
      }
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v = __builtin_amdgcn_mfma_f64_16x16x4f64(-d.l[16 * q + r16][16 * s + 4 * e + g], X[16 * s + 4 * e + g][r16], v, 0,
                                               0, 0);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) X[16 * q + 4 * i + g][r16] = v[i];
}

// X (64 rows x 16 columns in LDS, row stride 16) := T^-1 X by one wavefront: 16 rows by substitution
// (every 16-lane group alike; the first writes), their product subtracted from the remaining rows.
template <bool UPPER>
__device__ __forceinline__ void solve64_wave(double (*X)[16], const Diag64& d, int lane) {
  const int r16 = lane & 15, g = lane >> 4;
  const bool special = has_special(d);
#pragma unroll 1
  for (int s0 = 0; s0 < 4; ++s0) {
    const int s = UPPER ? 3 - s0 : s0;
    double x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = X[16 * s + i][r16];
    substitute16<UPPER>(x, d, s);
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    if (g == 0) {
#pragma unroll
      for (int i = 0; i < 16; ++i) X[16 * s + i][r16] = x[i];
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
#pragma unroll 1
    for (int q = UPPER ? 0 : s + 1; q < (UPPER ? s : 4); ++q) subtract_part16(X, d, q, s, special, lane);
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
  }
}

// ---- a factored panel's interchanges on every other column, and U12 -----------------------------
// 64 columns per workgroup, one per lane (a wavefront's row accesses are 512 contiguous bytes), 16
// rows per wavefront.  The panel's nb rows go to LDS; a row below the panel that takes part always
// receives one of them (a row of the panel not yet reached by the interchanges only ever holds a
// row of the panel), a row of the panel receives one of them or a row from below, read before
// anything is written.  The columns p0 + 64 .. solve_end - 1 then get U12 = L11^-1 A12 (full panels
// only: a partial panel is the matrix's last).  The columns on the left only exchange rows.  Panels
// start at multiples of 64, so a workgroup's columns lie on one side.
__global__ __launch_bounds__(256) void panel_swap_kernel(double* __restrict__ A, const double* __restrict__ L, long lda,
                                                         int n, int p0, int nb, int solve_end,
                                                         const int32_t* __restrict__ ipiv) {
  __shared__ Diag64 s_d;
  __shared__ double s_x[4][kPanel][16];  // column tile, row, column
  __shared__ int s_piv[kPanel], s_src[2 * kPanel];
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int ct = lane >> 4, cc = lane & 15;
  const long oc = (long)blockIdx.x * kPanel + lane;
  const bool on = oc < n - nb;
  const long oc1 = on ? oc : n - nb - 1;
  const long col = oc1 < p0 ? oc1 : oc1 + nb;
  const int first = blockIdx.x * kPanel;  // the workgroup's first column
  const bool solve = nb == kPanel && first >= p0 && first + nb < solve_end;
  if (t < kPanel) s_piv[t] = t < nb ? ipiv[p0 + t] - 1 : p0 + t;
  double x[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int r = 16 * wave + i;
    x[i] = r < nb ? A[(long)(p0 + r) * lda + col] : 0.0;
  }
  if (solve) load_diag64<false>(s_d, L + (long)p0 * lda + p0, lda, kPanel);
  __syncthreads();
  // sources of the panel's rows (first 64) and of the rows below that the interchanges touch
  if (t < 2 * kPanel) {
    const int q = t & 63, dst = t < kPanel ? p0 + q : s_piv[q];
    const bool use = q < nb && (t < kPanel || dst >= p0 + nb);
    s_src[t] = use ? swap_source(dst, s_piv, p0, nb) : -1;
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) s_x[ct][16 * wave + i][cc] = x[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int src = __builtin_amdgcn_readfirstlane(s_src[16 * wave + i]);
    if (src >= p0 + nb) x[i] = A[(long)src * lda + col];
    else if (src >= 0) x[i] = s_x[ct][src - p0][cc];
  }
  // every source row has been read before the first row is overwritten
  __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
#pragma unroll 1
  for (int i = 0; i < 16; ++i) {
    const int q = 16 * wave + i, src = __builtin_amdgcn_readfirstlane(s_src[kPanel + q]);
    if (src >= 0 && on) A[(long)s_piv[q] * lda + col] = s_x[ct][src - p0][cc];
  }
  if (solve) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) s_x[ct][16 * wave + i][cc] = x[i];
    __syncthreads();
    solve64_wave<false>(s_x[wave], s_d, lane);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = s_x[ct][16 * wave + i][cc];
    // (columns past solve_end in this workgroup: solve_end is a multiple of 64 or the matrix's end)
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int r = 16 * wave + i;
    if (on && r < nb) A[(long)(p0 + r) * lda + col] = x[i];
  }
}

// B (64 x ncols) := T^-1 B for a full 64 x 64 diagonal block, 64 columns per workgroup.
template <bool UPPER>
__global__ __launch_bounds__(256) void trsm64_kernel(const double* __restrict__ T, long ldt, double* __restrict__ B,
                                                     long ldb, long ncols) {
  __shared__ Diag64 s_d;
  __shared__ double s_x[4][kPanel][16];
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const long col = (long)blockIdx.x * kPanel + lane;
  const bool on = col < ncols;
  double x[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) x[i] = on ? B[(long)(16 * wave + i) * ldb + col] : 0.0;
  load_diag64<UPPER>(s_d, T, ldt, kPanel);
#pragma unroll
  for (int i = 0; i < 16; ++i) s_x[lane >> 4][16 * wave + i][lane & 15] = x[i];
  __syncthreads();
  solve64_wave<UPPER>(s_x[wave], s_d, lane);
  __syncthreads();
  if (on) {
#pragma unroll
    for (int i = 0; i < 16; ++i) B[(long)(16 * wave + i) * ldb + col] = s_x[lane >> 4][16 * wave + i][lane & 15];
  }
}

// ---- one block step of a triangular solve with few right-hand sides -----------------------------
// X(b0 .. b0 + nb - 1) = T_bb^-1 W(b0 ..), then W(rest) -= T(rest, b) X, rest = the rows below
// (lower) or above (upper); nb <= 64.  blockIdx.x: 64 of the remaining rows, blockIdx.y: 16
// columns.  Every workgroup solves the diagonal block for itself, so a block costs one launch;
// the solved rows go to X (written by the first workgroup), never over the rows of W that the
// other workgroups still read.  The block is solved by 16-row parts: one wavefront substitutes,
// the others subtract its part with FP64 MFMAs (the strip of T below or above is read before the
// solve, behind which its latency hides).
template <bool UPPER>
__global__ __launch_bounds__(256) void trsv_block_kernel(const double* __restrict__ T, long ldt, int n, int b0, int nb,
                                                         double* __restrict__ W, long ldw, double* __restrict__ X,
                                                         long ldx, int ncols, const int32_t* __restrict__ info) {
  __shared__ Diag64 s_d;
  __shared__ double s_x[kPanel][16];
  const int lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c0 = blockIdx.y * 16;
  const bool con = c0 + r16 < ncols;
  const int rest0 = UPPER ? 0 : b0 + nb, rest1 = UPPER ? b0 : n;
  const int row0 = rest0 + blockIdx.x * 64 + wave * 16;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int br = 16 * wave + 4 * i + g;
    s_x[br][r16] = (br < nb && con) ? W[(long)(b0 + br) * ldw + c0 + r16] : 0.0;
  }
  load_diag64<UPPER>(s_d, T + (long)b0 * ldt + b0, ldt, nb);
  // this wavefront's 16 remaining rows: columns 16 g .. 16 g + 15 of the block per lane, and the
  // tile of W
  double tr[16];
  d4 acc = {0.0, 0.0, 0.0, 0.0};
  const int rr = row0 + r16;
#pragma unroll
  for (int e = 0; e < 16; ++e) tr[e] = (rr < rest1 && 16 * g + e < nb) ? T[(long)rr * ldt + b0 + 16 * g + e] : 0.0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int wr = row0 + 4 * i + g;
    if (wr < rest1 && con) acc[i] = W[(long)wr * ldw + c0 + r16];
  }
  __syncthreads();
  const bool special = has_special(s_d);
#pragma unroll 1
  for (int s0 = 0; s0 < 4; ++s0) {
    const int s = UPPER ? 3 - s0 : s0;
    if (wave == s) {  // every 16-lane group substitutes alike; the first writes
      double x[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) x[i] = s_x[16 * s + i][r16];
      substitute16<UPPER>(x, s_d, s);
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
      if (g == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) s_x[16 * s + i][r16] = x[i];
      }
    }
    __syncthreads();
    if (UPPER ? wave < s : wave > s) {
      subtract_part16(s_x, s_d, wave, s, special, lane);
      // the wavefront that substitutes next reads, in each lane, what its other lanes wrote here
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    }
  }
  // after the last part nothing is updated: s_x is final
#pragma unroll
  for (int e = 0; e < 16; ++e)
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-tr[e], s_x[16 * g + e][r16], acc, 0, 0, 0);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int wr = row0 + 4 * i + g;
    if (wr < rest1 && con) W[(long)wr * ldw + c0 + r16] = acc[i];
  }
  if (blockIdx.x == 0 && con && (info == nullptr || *info == 0)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int br = 16 * wave + 4 * i + g;
      if (br < nb) X[(long)(b0 + br) * ldx + c0 + r16] = s_x[br][r16];
    }
  }
}

// ---- triangular solves on 32 x 32 diagonal blocks ---------------------------------------------
// B (nb x ncols, nb <= 32) := T^-1 B, T lower unit (UPPER = false) or upper non-unit, one
// thread per column; the operation order of reference dtrsm (Left, NoTrans): for each k in
// order, skip a zero B(k), scale by the diagonal (upper), subtract B(k) T(i, k) from the rest.
template <bool UPPER>
__global__ __launch_bounds__(256) void trsm_leaf_kernel(const double* __restrict__ T, long ldt, int nb,
                                                        double* __restrict__ B, long ldb, long ncols) {
  __shared__ double sT[kTrsmLeaf][kTrsmLeaf + 1];
  for (int e = threadIdx.x; e < nb * nb; e += 256) sT[e / nb][e % nb] = T[(long)(e / nb) * ldt + e % nb];
  __syncthreads();
  const long col = (long)blockIdx.x * 256 + threadIdx.x;
  if (col >= ncols) return;
  double x[kTrsmLeaf];
#pragma unroll
  for (int i = 0; i < kTrsmLeaf; ++i) x[i] = i < nb ? B[(long)i * ldb + col] : 0.0;
  if (!UPPER) {
#pragma unroll
    for (int k = 0; k < kTrsmLeaf; ++k) {
      if (k < nb && x[k] != 0.0) {
#pragma unroll
        for (int i = k + 1; i < kTrsmLeaf; ++i)
          if (i < nb) x[i] -= x[k] * sT[i][k];
      }
    }
  } else {
#pragma unroll
    for (int k = kTrsmLeaf - 1; k >= 0; --k) {
      if (k < nb && x[k] != 0.0) {
        x[k] = x[k] / sT[k][k];
#pragma unroll
        for (int i = 0; i < k; ++i) x[i] -= x[k] * sT[i][k];
      }
    }
  }
#pragma unroll
  for (int i = 0; i < kTrsmLeaf; ++i)
    if (i < nb) B[(long)i * ldb + col] = x[i];
}

// ---- row permutation of the right-hand sides ---------------------------------------------------
// For every 64 interchanges (one workgroup of 128 threads), the net move of the at most 128
// positions they touch: move[128 b + t] = (destination, source), destination -1 for none.  Factors
// from elsewhere may interchange a row with any other, also with one above its block.
__global__ __launch_bounds__(128) void ipiv_moves_kernel(int n, const int32_t* __restrict__ ipiv,
                                                         int2* __restrict__ moves) {
  __shared__ int s_piv[kPanel];
  const int t = threadIdx.x, base = blockIdx.x * kPanel, w = min(kPanel, n - base);
  if (t < kPanel) s_piv[t] = t < w ? ipiv[base + t] - 1 : base + t;
  __syncthreads();
  const int q = t % kPanel;
  int dst = -1;
  if (q < w) dst = t < kPanel ? base + q : s_piv[q];
  if (t >= kPanel && dst >= base && dst < base + w) dst = -1;
  moves[(long)blockIdx.x * 128 + t] = make_int2(dst, dst >= 0 ? swap_source(dst, s_piv, base, w) : -1);
}

// perm[i] = the original row that ends at position i after the interchanges ipiv[0..n) in
// order: the blocks of moves applied one after another in LDS (n <= kMaxOrder, one workgroup).
// 64 interchanges cost two barriers; one thread following them one by one took 83 ns each
// (n = 3000: 248 us).
__global__ __launch_bounds__(128) void moves_to_perm_kernel(int n, const int2* __restrict__ moves,
                                                            int32_t* __restrict__ perm) {
  extern __shared__ int sp[];
  const int t = threadIdx.x, nblk = (n + kPanel - 1) / kPanel;
  for (int i = t; i < n; i += 128) sp[i] = i;
  int2 cur = moves[t];
  __syncthreads();
  for (int b = 0; b < nblk; ++b) {
    int2 next = cur;
    if (b + 1 < nblk) next = moves[(long)(b + 1) * 128 + t];
    const int v = cur.x >= 0 ? sp[cur.y] : 0;
    __syncthreads();
    if (cur.x >= 0) sp[cur.x] = v;
    __syncthreads();
    cur = next;
  }
  for (int i = t; i < n; i += 128) perm[i] = sp[i];
}

// perm of up to 64 interchanges in one launch: each position traced back by itself.
__global__ __launch_bounds__(64) void ipiv_to_perm64_kernel(int n, const int32_t* __restrict__ ipiv,
                                                            int32_t* __restrict__ perm) {
  __shared__ int s_piv[kPanel];
  const int t = threadIdx.x;
  s_piv[t] = t < n ? ipiv[t] - 1 : t;
  __syncthreads();
  if (t < n) perm[t] = swap_source(t, s_piv, 0, n);
}

// W[i][c] = B[perm[i]][c] (identity = true: W = P I, the permuted identity, n x n)
__global__ __launch_bounds__(256) void gather_rows_kernel(int n, long ncols, const int32_t* __restrict__ perm,
                                                          const double* __restrict__ B, long ldb,
                                                          double* __restrict__ W, long ldw, bool identity) {
  const long e = (long)blockIdx.x * 256 + threadIdx.x;
  if (e >= (long)n * ncols) return;
  const long i = e / ncols, c = e % ncols;
  const int src = perm[i];
  W[i * ldw + c] = identity ? (src == c ? 1.0 : 0.0) : B[(long)src * ldb + c];
}

// B = W, unless info is given and nonzero
__global__ __launch_bounds__(256) void copy_rows_kernel(int n, long ncols, const double* __restrict__ W, long ldw,
                                                        double* __restrict__ B, long ldb,
                                                        const int32_t* __restrict__ info) {
  const long e = (long)blockIdx.x * 256 + threadIdx.x;
  if (e >= (long)n * ncols || (info != nullptr && *info != 0)) return;
  const long i = e / ncols, c = e % ncols;
  B[i * ldb + c] = W[i * ldw + c];
}

__global__ void zero_info_kernel(int32_t* info) { *info = 0; }

// detNxN's rule from the factors: 0 for a zero pivot, else the product, left to right from 1,
// of U's diagonal with the sign flipped at every interchange.
__global__ void det_kernel(int n, const double* __restrict__ A, long lda, const int32_t* __restrict__ ipiv,
                           const int32_t* __restrict__ info, double* __restrict__ out) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  if (*info > 0) {
    *out = 0.0;
    return;
  }
  double d = 1.0;
  for (int i = 0; i < n; ++i) {
    d *= A[(long)i * lda + i];
    if (ipiv[i] != i + 1) d = -d;
  }
  *out = d;
}

// ---- host side -------------------------------------------------------------------------------
// threads, rows per thread and leaf width for a panel of m rows: one wavefront per SIMD while its
// registers hold 16 columns of the block, then two, then fewer columns.  The smallest matrices (and a last
// panel's end) take half the column loop: n = 1 10.8 us, 15.3 with the 16-column leaf; n = 8 13.0, 20.6.
struct LeafShape {
  int t, r, wl;
};
static LeafShape leaf_shape(int64_t m) {
  if (m <= 8) return {256, 1, 8};
  static const LeafShape shapes[] = {{256, 1, 16}, {256, 2, 16}, {256, 4, 16}, {256, 6, 16}, {512, 4, 16},
                                     {512, 6, 12}, {512, 8, 8},  {512, 16, 4}, {512, 32, 2}, {512, 64, 1}};
  for (const LeafShape& s : shapes)
    if ((int64_t)s.t * s.r >= m) return s;
  return {0, 0, 0};
}

// Factors the leaf c0 .. c0 + w - 1 of the panel p0 .. p0 + nbp - 1 and subtracts its product from
// the panel's columns on its right.
static bzg_status launch_leaf(bzg_context* ctx, double* A, long lda, int n, int c0, int w, int p0, int nbp,
                              int32_t* ipiv, int32_t* info) {
  const LeafShape sh = leaf_shape(n - c0);
  const int r0 = c0 + w, nc = p0 + nbp - r0, rows = n - r0;
  const unsigned ugrid = (unsigned)((rows + 4 * kRankRows - 1) / (4 * kRankRows));
#define BZG_LEAF(TT, RR, WW)                                                                               \
  if (sh.t == TT && sh.r == RR && sh.wl == WW) {                                                           \
    hipLaunchKernelGGL((getf2_leaf_kernel<TT, RR, WW>), dim3(1), dim3(TT), 0, ctx->stream, A, lda, n, c0, w, p0, nbp, \
                       ipiv, info);                                                                        \
    BZG_LAUNCH_CHECK();                                                                                    \
    if (nc > 0 && rows > 0) { /* w == WW here: only the panel's last leaf is narrower */                   \
      hipLaunchKernelGGL((rank_update_kernel<WW>), dim3(ugrid), dim3(256), 0, ctx->stream, A, A, A, lda, n, r0, nc); \
      BZG_LAUNCH_CHECK();                                                                                  \
    }                                                                                                      \
    return BZG_OK;                                                                                         \
  }
  BZG_LEAF(256, 1, 8)
  BZG_LEAF(256, 1, 16)
  BZG_LEAF(256, 2, 16)
  BZG_LEAF(256, 4, 16)
  BZG_LEAF(256, 6, 16)
  BZG_LEAF(512, 4, 16)
  BZG_LEAF(512, 6, 12)
  BZG_LEAF(512, 8, 8)
  BZG_LEAF(512, 16, 4)
  BZG_LEAF(512, 32, 2)
  BZG_LEAF(512, 64, 1)
#undef BZG_LEAF
  set_error("getrf: panel taller than 32768 rows");
  return BZG_ERR_UNSUPPORTED;
}

// B (nb x ncols) := T^-1 B with T the nb x nb diagonal block at T (lower unit or upper).
static bzg_status trsm(bzg_context* ctx, bool upper, const double* T, long ldt, int nb, double* B, long ldb,
                       long ncols) {
  if (nb <= 0 || ncols <= 0) return BZG_OK;
  if (nb == kPanel) {
    const unsigned grid = (unsigned)((ncols + 63) / 64);
    if (upper)
      hipLaunchKernelGGL(trsm64_kernel<true>, dim3(grid), dim3(256), 0, ctx->stream, T, ldt, B, ldb, ncols);
    else
      hipLaunchKernelGGL(trsm64_kernel<false>, dim3(grid), dim3(256), 0, ctx->stream, T, ldt, B, ldb, ncols);
    BZG_LAUNCH_CHECK();
    return BZG_OK;
  }
  if (nb <= kTrsmLeaf) {
    const unsigned grid = (unsigned)((ncols + 255) / 256);
    if (upper)
      hipLaunchKernelGGL(trsm_leaf_kernel<true>, dim3(grid), dim3(256), 0, ctx->stream, T, ldt, nb, B, ldb, ncols);
    else
      hipLaunchKernelGGL(trsm_leaf_kernel<false>, dim3(grid), dim3(256), 0, ctx->stream, T, ldt, nb, B, ldb, ncols);
    BZG_LAUNCH_CHECK();
    return BZG_OK;
  }
  // split at a multiple of 64 (of 32 below 64)
  const int q = nb > kPanel ? kPanel : kTrsmLeaf;
  const int h = std::max(q, nb / 2 / q * q);
  bzg_status st;
  if (!upper) {
    // [L11 0; L21 L22]: X1 = L11^-1 B1, B2 -= L21 X1, X2 = L22^-1 B2
    if ((st = trsm(ctx, false, T, ldt, h, B, ldb, ncols))) return st;
    if ((st = bzg_dgemm(ctx, nb - h, ncols, h, -1.0, T + (long)h * ldt, ldt, B, ldb, 1.0, B + (long)h * ldb, ldb)))
      return st;
    return trsm(ctx, false, T + (long)h * ldt + h, ldt, nb - h, B + (long)h * ldb, ldb, ncols);
  }
  // [U11 U12; 0 U22]: X2 = U22^-1 B2, B1 -= U12 X2, X1 = U11^-1 B1
  if ((st = trsm(ctx, true, T + (long)h * ldt + h, ldt, nb - h, B + (long)h * ldb, ldb, ncols))) return st;
  if ((st = bzg_dgemm(ctx, h, ncols, nb - h, -1.0, T + h, ldt, B + (long)h * ldb, ldb, 1.0, B, ldb))) return st;
  return trsm(ctx, true, T, ldt, h, B, ldb, ncols);
}

// Columns up to which a block is factored panel by panel (rank-64 updates of everything on the
// right); wider blocks are split in half, so that their updates have more work per byte.
constexpr int kRightLooking = 2048;

// Factors columns d0 .. d0 + nc - 1 on rows d0 .. n - 1 (d0 a multiple of 64), interchanges applied
// to every column of the matrix.
static bzg_status rgetrf(bzg_context* ctx, double* A, long lda, int n, int d0, int nc, int32_t* ipiv,
                         int32_t* info) {
  bzg_status st;
  if (nc > kRightLooking) {  // dgetrf2's recursion
    const int n1 = (nc / 2 + kPanel - 1) / kPanel * kPanel, n2 = nc - n1, m = n - d0;
    if ((st = rgetrf(ctx, A, lda, n, d0, n1, ipiv, info))) return st;
    double* A11 = A + (long)d0 * lda + d0;
    // U12 = L11^-1 A12, then A22 -= L21 U12
    if ((st = trsm(ctx, false, A11, lda, n1, A11 + n1, lda, n2))) return st;
    if ((st = bzg_dgemm(ctx, m - n1, n2, n1, -1.0, A11 + (long)n1 * lda, lda, A11 + n1, lda, 1.0,
                        A11 + (long)n1 * lda + n1, lda)))
      return st;
    return rgetrf(ctx, A, lda, n, d0 + n1, n2, ipiv, info);
  }
  const int end = d0 + nc;
  for (int p0 = d0; p0 < end; p0 += kPanel) {
    const int nbp = std::min(kPanel, end - p0);
    for (int c0 = p0; c0 < p0 + nbp;) {
      const int w = std::min(leaf_shape(n - c0).wl, p0 + nbp - c0);
      if ((st = launch_leaf(ctx, A, lda, n, c0, w, p0, nbp, ipiv, info))) return st;
      c0 += w;
    }
    if (n == nbp) return BZG_OK;  // no other columns
    hipLaunchKernelGGL(panel_swap_kernel, dim3((unsigned)((n - nbp + kPanel - 1) / kPanel)), dim3(256), 0, ctx->stream, A,
                       A, lda, n, p0, nbp, end, ipiv);
    BZG_LAUNCH_CHECK();
    const int r0 = p0 + nbp;
    if (r0 < end && r0 < n) {
      double* A22 = A + (long)r0 * lda + r0;
      if ((st = bzg_dgemm(ctx, n - r0, end - r0, nbp, -1.0, A22 - nbp, lda, A22 - (long)nbp * lda, lda, 1.0, A22, lda)))
        return st;
    }
  }
  return BZG_OK;
}

static bzg_status check_square(bzg_context* ctx, int64_t n, const void* A, int64_t lda, const char* what) {
  if (!ctx) {
    set_error(std::string(what) + ": null context");
    return BZG_ERR_INVALID_ARGUMENT;
  }
  if (n < 0 || lda < (n > 0 ? n : 1)) {
    set_error(std::string(what) + ": bad order or leading dimension");
    return BZG_ERR_INVALID_ARGUMENT;
  }
  if (n > kMaxOrder) {
    set_error(std::string(what) + ": order above 32768");
    return BZG_ERR_UNSUPPORTED;
  }
  if (n > 0 && !A) {
    set_error(std::string(what) + ": null matrix");
    return BZG_ERR_INVALID_ARGUMENT;
  }
  return BZG_OK;
}

// The permutation kernel's LDS (4 bytes per row) beyond 64 KB needs the attribute raised once per
// device.
static std::mutex g_perm_mu;
static bool g_perm_attr[64] = {};

static bzg_status perm_attr(bzg_context* ctx) {
  if (ctx->device < 0 || ctx->device >= 64) return BZG_OK;
  std::lock_guard<std::mutex> lock(g_perm_mu);
  if (g_perm_attr[ctx->device]) return BZG_OK;
  BZG_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&moves_to_perm_kernel),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)(kMaxOrder * sizeof(int))));
  g_perm_attr[ctx->device] = true;
  return BZG_OK;
}

// Right-hand sides up to which a triangular solve runs block by block (trsv_block_kernel); more
// go through the recursion and bzg_dgemm, and so do matrices with fewer rows than this: there a thread
// solves a column by itself (n = 12, 16 right-hand sides: 20.8 us, 22.7 by blocks; 20, 17: 24.6, 27.1; alike
// at 24).
constexpr long kBlockSolveCols = 64;
constexpr int kBlockSolveRows = 25;

// B := A^-1 B (B := A^-1 when identity) from the factors, unless info is given and nonzero:
// W = P B (or P I) in the context's workspaces, forward and back substitution.
static bzg_status getrs_run(bzg_context* ctx, int n, long ncols, const double* LU, long lda, const int32_t* ipiv,
                            double* B, long ldb, bool identity, const int32_t* info) {
  // (the inverse replaces the factors, which the block solve still reads when it writes B)
  const bool blocks = !identity && ncols <= kBlockSolveCols && n >= kBlockSolveRows;
  const int nblk = (n + kPanel - 1) / kPanel;
  // slot 13: the interchanges' moves and perm; slot 14: W and, for the block solve, the forward
  // solution
  void *p = nullptr, *w = nullptr;
  bzg_status st = workspace(ctx, 13, (size_t)nblk * 128 * sizeof(int2) + (size_t)n * sizeof(int32_t), &p);
  if (!st) st = workspace(ctx, 14, (size_t)n * (size_t)ncols * sizeof(double) * (blocks ? 2 : 1), &w);
  if (!st) st = perm_attr(ctx);
  if (st) return st;
  int2* moves = static_cast<int2*>(p);
  int32_t* perm = reinterpret_cast<int32_t*>(moves + (size_t)nblk * 128);
  double* W = static_cast<double*>(w);
  if (nblk == 1) {  // (a launch less: n = 12, 65 right-hand sides 20.9 us, 24.1)
    hipLaunchKernelGGL(ipiv_to_perm64_kernel, dim3(1), dim3(64), 0, ctx->stream, n, ipiv, perm);
    BZG_LAUNCH_CHECK();
  } else {
    hipLaunchKernelGGL(ipiv_moves_kernel, dim3((unsigned)nblk), dim3(128), 0, ctx->stream, n, ipiv, moves);
    BZG_LAUNCH_CHECK();
    hipLaunchKernelGGL(moves_to_perm_kernel, dim3(1), dim3(128), (size_t)n * sizeof(int), ctx->stream, n, moves, perm);
    BZG_LAUNCH_CHECK();
  }
  const long total = (long)n * ncols;
  hipLaunchKernelGGL(gather_rows_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, ctx->stream, n, ncols,
                     perm, B, ldb, W, ncols, identity);
  BZG_LAUNCH_CHECK();
  if (blocks) {
    double* Y = W + (size_t)total;
    const unsigned gy = (unsigned)((ncols + 15) / 16);
    for (int b0 = 0; b0 < n; b0 += kPanel) {
      const int nb = std::min(kPanel, n - b0), rest = n - b0 - nb;
      hipLaunchKernelGGL(trsv_block_kernel<false>, dim3((unsigned)std::max(1, (rest + 63) / 64), gy), dim3(256), 0,
                         ctx->stream, LU, lda, n, b0, nb, W, ncols, Y, ncols, (int)ncols, (const int32_t*)nullptr);
      BZG_LAUNCH_CHECK();
    }
    for (int b0 = (nblk - 1) * kPanel; b0 >= 0; b0 -= kPanel) {
      const int nb = std::min(kPanel, n - b0);
      hipLaunchKernelGGL(trsv_block_kernel<true>, dim3((unsigned)std::max(1, (b0 + 63) / 64), gy), dim3(256), 0,
                         ctx->stream, LU, lda, n, b0, nb, Y, ncols, B, ldb, (int)ncols, info);
      BZG_LAUNCH_CHECK();
    }
    return BZG_OK;
  }
  if ((st = trsm(ctx, false, LU, lda, n, W, ncols, ncols))) return st;
  if ((st = trsm(ctx, true, LU, lda, n, W, ncols, ncols))) return st;
  hipLaunchKernelGGL(copy_rows_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, ctx->stream, n, ncols, W,
                     ncols, B, ldb, info);
  BZG_LAUNCH_CHECK();
  return BZG_OK;
}

}  // namespace big
}  // namespace bzg

extern "C" {

bzg_status bzg_dgetrf(bzg_context* ctx, int64_t n, double* A, int64_t lda, int32_t* ipiv, int32_t* info) {
  bzg_status st = bzg::big::check_square(ctx, n, A, lda, "dgetrf");
  if (st) return st;
  BZG_REQUIRE(info != nullptr && (n == 0 || ipiv != nullptr), BZG_ERR_INVALID_ARGUMENT, "dgetrf: null ipiv or info");
  bzg::ProfScope prof(ctx, "dgetrf");
  hipLaunchKernelGGL(bzg::big::zero_info_kernel, dim3(1), dim3(1), 0, ctx->stream, info);
  BZG_LAUNCH_CHECK();
  if (n == 0) return BZG_OK;
  return bzg::big::rgetrf(ctx, A, (long)lda, (int)n, 0, (int)n, ipiv, info);
}

bzg_status bzg_dgetrs(bzg_context* ctx, int64_t n, int64_t nrhs, const double* A, int64_t lda,
                      const int32_t* ipiv, double* B, int64_t ldb) {
  bzg_status st = bzg::big::check_square(ctx, n, A, lda, "dgetrs");
  if (st) return st;
  BZG_REQUIRE(nrhs >= 0 && ldb >= (nrhs > 0 ? nrhs : 1), BZG_ERR_INVALID_ARGUMENT, "dgetrs: bad nrhs or ldb");
  if (n == 0 || nrhs == 0) return BZG_OK;
  BZG_REQUIRE(ipiv != nullptr && B != nullptr, BZG_ERR_INVALID_ARGUMENT, "dgetrs: null ipiv or B");
  bzg::ProfScope prof(ctx, "dgetrs");
  return bzg::big::getrs_run(ctx, (int)n, (long)nrhs, A, (long)lda, ipiv, B, (long)ldb, false, nullptr);
}

bzg_status bzg_dgesv(bzg_context* ctx, int64_t n, int64_t nrhs, double* A, int64_t lda, int32_t* ipiv, double* B,
                     int64_t ldb, int32_t* info) {
  bzg_status st = bzg::big::check_square(ctx, n, A, lda, "dgesv");
  if (st) return st;
  BZG_REQUIRE(nrhs >= 0 && ldb >= (nrhs > 0 ? nrhs : 1), BZG_ERR_INVALID_ARGUMENT, "dgesv: bad nrhs or ldb");
  if ((st = bzg_dgetrf(ctx, n, A, lda, ipiv, info))) return st;
  if (n == 0 || nrhs == 0) return BZG_OK;
  // dgesv leaves B unchanged when the factorisation reports a zero pivot: the kernels that write B
  // read info on the device
  if (B != nullptr) {
    bzg::ProfScope prof(ctx, "dgetrs");
    st = bzg::big::getrs_run(ctx, (int)n, (long)nrhs, A, (long)lda, ipiv, B, (long)ldb, false, info);
    if (st != BZG_ERR_OUT_OF_MEMORY) return st;
  } else {
    bzg::set_error("dgesv: null B");
    st = BZG_ERR_INVALID_ARGUMENT;
  }
  // a singular matrix needs neither B nor the solve's scratch: only then is info read back
  int32_t h_info = 0;
  BZG_HIP_CHECK(hipMemcpyAsync(&h_info, info, sizeof(int32_t), hipMemcpyDeviceToHost, ctx->stream));
  BZG_HIP_CHECK(hipStreamSynchronize(ctx->stream));
  return h_info != 0 ? BZG_OK : st;
}

bzg_status bzg_dgetri(bzg_context* ctx, int64_t n, double* A, int64_t lda, const int32_t* ipiv) {
  bzg_status st = bzg::big::check_square(ctx, n, A, lda, "dgetri");
  if (st) return st;
  if (n == 0) return BZG_OK;
  BZG_REQUIRE(ipiv != nullptr, BZG_ERR_INVALID_ARGUMENT, "dgetri: null ipiv");
  bzg::ProfScope prof(ctx, "dgetri");
  return bzg::big::getrs_run(ctx, (int)n, (long)n, A, (long)lda, ipiv, A, (long)lda, true, nullptr);
}

bzg_status bzg_ddet_lu(bzg_context* ctx, int64_t n, const double* A, int64_t lda, const int32_t* ipiv,
                       const int32_t* info, double* det) {
  bzg_status st = bzg::big::check_square(ctx, n, A, lda, "ddet_lu");
  if (st) return st;
  BZG_REQUIRE(info != nullptr && det != nullptr && (n == 0 || ipiv != nullptr), BZG_ERR_INVALID_ARGUMENT,
              "ddet_lu: null ipiv, info or det");
  hipLaunchKernelGGL(bzg::big::det_kernel, dim3(1), dim3(64), 0, ctx->stream, (int)n, A, (long)lda, ipiv, info, det);
  BZG_LAUNCH_CHECK();
  return BZG_OK;
}

}  // extern "C"
