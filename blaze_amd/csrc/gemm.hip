// Dense GEMM for gfx950:  C = alpha * A * B + beta * C, row-major operands.
//
// Replaces the assignment kernels of DMatDMatMultExpr (blaze/math/expressions/
// DMatDMatMultExpr.h:516-569 dispatch, :864-1887 small kernel, MMM.h:105-600 blocked kernel).
//
// FP64 / FP32: MFMA 16x16x4 tiles (v_mfma_f64_16x16x4f64, v_mfma_f32_16x16x4f32).  A workgroup
// of 4 wavefronts computes a BM x BN tile of C; each wave owns a WM x WN sub-tile held in
// MFMA accumulators.  A and B K-slabs of depth BK are staged through LDS with two buffers:
// global loads of the next slab (small tiles: the next two) are in flight in registers during the
// MFMAs of a slab and written to the idle LDS buffer afterwards, so one barrier per slab suffices.
// Small tiles are bound by that latency, so their slabs are deep (256 bytes of k for 32 x 32, 128 for
// 64 x 64): 512^3 FP64 9.7 us = 27.7 TFLOP/s (22.7 us with 16 of k, one slab ahead), 1024^3 FP32
// 27 us (39.8), 1523 x 1777 x 2021 FP32 with odd leading dimensions 100 us (181: 4-byte loads).
// Large tiles are bound by the matrix cores: 4096^3 68.2 TFLOP/s FP64, 134 FP32.
// Every C element is produced by one wave in a fixed k order (no split-K, no atomics), so the
// result is identical run to run and independent of the launch shape chosen for other calls.
//
// INT32: no integer MFMA takes 32-bit operands; a VALU kernel with LDS tiles and 4x4 register
// micro-tiles in wrap-around uint32 arithmetic (bit-exact against any summation order).
#include "common.hpp"

#include <algorithm>
#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>

namespace bzg {
namespace {

constexpr int kThreads = 256;

template <typename T>
struct Mfma;

template <>
struct Mfma<double> {
  using acc_t = d4;
  __device__ static acc_t mma(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  // Accumulator register i of lane l holds row 4*i + l/16, column l%16 (measured on gfx950).
  __device__ static int row(int i, int lane) { return 4 * i + lane / 16; }
};

template <>
struct Mfma<float> {
  using acc_t = f4;
  __device__ static acc_t mma(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  // Accumulator register i of lane l holds row 4*(l/16) + i, column l%16.
  __device__ static int row(int i, int lane) { return 4 * (lane / 16) + i; }
};

// 16 bytes of elements, element-aligned: gfx950 takes a 16-byte global access at any element address
template <typename T>
struct Vec16;
template <>
struct Vec16<double> {
  typedef double type __attribute__((ext_vector_type(2), aligned(8)));
  typedef double aligned_type __attribute__((ext_vector_type(2)));
};
template <>
struct Vec16<float> {
  typedef float type __attribute__((ext_vector_type(4), aligned(4)));
  typedef float aligned_type __attribute__((ext_vector_type(4)));
};

// Maps the linear workgroup id to a (tile_m, tile_n) pair.  Consecutive workgroup ids are
// dispatched round-robin over the 8 XCDs; the remap gives each XCD a contiguous range of
// logical tiles, and logical tiles are walked in column-major groups of 8 tile rows so the
// workgroups resident on one XCD share A row panels and B column panels in that XCD's L2.
__device__ __forceinline__ void tile_coords(int tiles_m, int tiles_n, int& tm, int& tn) {
  const int nt = tiles_m * tiles_n;
  int bid = blockIdx.x;
  int logical = bid;
  if (nt >= 64 && (nt % 8) == 0) logical = (bid % 8) * (nt / 8) + bid / 8;
  constexpr int G = 8;
  const int group = logical / (G * tiles_n);
  const int first_m = group * G;
  const int gsize = min(tiles_m - first_m, G);
  const int in_group = logical % (G * tiles_n);
  tm = first_m + in_group % gsize;
  tn = in_group / gsize;
}

// A slab stored [BM][BK + pad], B slab [BK][BN + pad].  Strides for which the fragment reads hit
// distinct banks (A: 4 banks modulo 64 from row to row; B: rows k and k + 1 half the banks apart) and
// rows start 16-byte aligned for vector stores.  A transposed operand is stored element by
// element along the other direction: there the strides are 1 modulo 16 elements, so that the
// rows a wavefront writes at once spread over 16 banks instead of 8 (A) or 1 (B).
template <typename T, int BM, int BN, int BK, bool TA = false, bool TB = false>
struct GemmShm {
  static constexpr int LDA = TA ? (BK + 16) / 32 * 32 + 17 - (BK % 32 ? 32 : 0) : BK + 16 / (int)sizeof(T);
  static constexpr int LDB = BN + (TB ? 17 : 16);
  __align__(16) T As[2][BM * LDA];
  __align__(16) T Bs[2][BK * LDB];
};

// One BM x BN tile (tm, tn) of C = alpha A B + beta C by the 4 wavefronts of the workgroup.
// Every element of C is summed in the same k order (MFMA k-steps of 4) whatever the tile shape
// and slab depth, so all tile shapes give bit-identical results.
// TA / TB: A (B) is given transposed, i.e. stored k x m (n x k) row-major with leading
// dimension lda >= m (ldb >= k); the slabs are then read along m (k) and transposed on the
// way into LDS, so the MFMA loop and its summation order are the same for all four forms.
//
// PF slabs of global loads are in flight in registers ahead of the slab being multiplied.
// The loads are 16 bytes at element alignment (odd leading dimensions take the same path).  Rows
// past the matrix are read as its last row and columns past it as its last column: they feed
// only elements of C that are not stored.  Only the last slab, if K is not a multiple of BK,
// checks k (and is zero beyond K in both operands).
template <typename T, int BM, int BN, int WM, int WN, int BK, int PF, bool TA = false, bool TB = false>
__device__ __forceinline__ void gemm_tile(int M, int N, int K, T alpha, const T* __restrict__ A,
                                          long lda, const T* __restrict__ B, long ldb, T beta,
                                          T* __restrict__ C, long ldc, int tm, int tn,
                                          GemmShm<T, BM, BN, BK, TA, TB>& sh) {
  using MF = Mfma<T>;
  using acc_t = typename MF::acc_t;
  using VU = typename Vec16<T>::type;          // 16 bytes, element-aligned (global memory)
  using VA = typename Vec16<T>::aligned_type;  // 16-byte aligned (LDS)
  constexpr int VW = 16 / (int)sizeof(T);
  constexpr int WAVES_N = BN / WN;
  constexpr int FM = WM / 16;  // MFMA blocks per wave along m
  constexpr int FN = WN / 16;  // MFMA blocks per wave along n
  constexpr int LDA_S = GemmShm<T, BM, BN, BK, TA, TB>::LDA;
  constexpr int LDB_S = GemmShm<T, BM, BN, BK, TA, TB>::LDB;
  constexpr int NA = BM * BK / (VW * kThreads);  // vectors per thread, A slab
  constexpr int NB = BK * BN / (VW * kThreads);  // vectors per thread, B slab
  // stored rows of a slab: A [m][k] (TA: [k][m]), B [k][n] (TB: [n][k]); vectors per stored row and
  // stored rows per pass of the workgroup
  constexpr int A_VPR = (TA ? BM : BK) / VW, A_RPP = kThreads / A_VPR;
  constexpr int B_VPR = (TB ? BK : BN) / VW, B_RPP = kThreads / B_VPR;
  static_assert(NA >= 1 && NB >= 1, "tile too small for 256 threads");
  static_assert((BM / WM) * (BN / WN) == 4, "four wavefronts per workgroup");
  static_assert(PF == 1 || PF == 2, "one or two slabs ahead");

  auto& As = sh.As;
  auto& Bs = sh.Bs;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm0 = (wave / WAVES_N) * WM;
  const int wn0 = (wave % WAVES_N) * WN;

  // Where an operand's stored rows run along m (A transposed) or n (B not), the matrix's last tile starts early
  // enough to be whole and stores only what its neighbour does not: all its loads stay vectors.  Read
  // element by element, such tiles were the last to end (2000^3 FP64, A transposed: 349 us, 259; 1000^3
  // FP32: 41.3, 29.6; 412 x 346, k = 111 FP32: 5.2, 4.6).
  const int m0 = TA && M >= BM ? min(tm * BM, M - BM) : tm * BM;
  const int n0 = !TB && N >= BN ? min(tn * BN, N - BN) : tn * BN;

  acc_t acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = acc_t{};

  struct Regs {
    VU a[NA], b[NB];
  };

  // One slab of both operands.  A stored row or column outside its matrix is read as the last one
  // (an address, never a selection: a selection would wait for the load); what lies beyond K is
  // zeroed on the way into LDS.
  const bool vec_a = !TA || m0 + BM <= M, vec_b = TB || n0 + BN <= N;
  auto load_op = [&](auto rows_k, bool vec, const T* __restrict__ X, long ldx, int o0, int lim, int k0, int r0, int c0,
                     VU& v) __attribute__((always_inline)) {
    constexpr bool ROWS_K = decltype(rows_k)::value;  // stored rows run along k
    if (vec) {
      const long row = ROWS_K ? r0 : min(o0 + r0, lim - 1);
      const T* p = X + row * ldx + (ROWS_K ? o0 + c0 : c0);
      v = *reinterpret_cast<const VU*>(p + (ROWS_K ? (long)k0 * ldx : (long)k0));
    } else {
      const int row = min((ROWS_K ? k0 : o0) + r0, (ROWS_K ? K : lim) - 1);
      const int col = (ROWS_K ? o0 : k0) + c0, cmax = (ROWS_K ? lim : K) - 1;
      const T* p = X + (long)row * ldx;
#pragma unroll
      for (int e = 0; e < VW; ++e) v[e] = p[min(col + e, cmax)];
    }
  };
  // `fast`: the slab is full and both operands are read by vectors, known at compile time.  SHALLOW tiles
  // often have no other slab than a partial one: where its rows run along k, those past K are read as the
  // last one, by vectors (3000 x 1000, k = 10 FP32, A transposed: 6.6 us, 7.3).
  constexpr bool SHALLOW = BM == 64 && PF == 1;
  auto load_slab = [&](auto fast, int k0, Regs& r) __attribute__((always_inline)) {
    constexpr bool FAST = decltype(fast)::value;
    const bool kfull = k0 + BK <= K;
    const bool va = FAST || (vec_a && kfull), vb = FAST || (vec_b && kfull);  // uniform
    if (va) {
#pragma unroll
      for (int i = 0; i < NA; ++i)
        load_op(std::integral_constant<bool, TA>{}, true, A, lda, m0, M, k0, tid / A_VPR + i * A_RPP, (tid % A_VPR) * VW,
                r.a[i]);
    } else if (SHALLOW && TA && vec_a) {
#pragma unroll
      for (int i = 0; i < NA; ++i)
        load_op(std::integral_constant<bool, TA>{}, true, A, lda, m0, M, k0, min(tid / A_VPR + i * A_RPP, K - 1 - k0),
                (tid % A_VPR) * VW, r.a[i]);
    } else {
#pragma unroll
      for (int i = 0; i < NA; ++i)
        load_op(std::integral_constant<bool, TA>{}, false, A, lda, m0, M, k0, tid / A_VPR + i * A_RPP,
                (tid % A_VPR) * VW, r.a[i]);
    }
    if (vb) {
#pragma unroll
      for (int i = 0; i < NB; ++i)
        load_op(std::integral_constant<bool, !TB>{}, true, B, ldb, n0, N, k0, tid / B_VPR + i * B_RPP,
                (tid % B_VPR) * VW, r.b[i]);
    } else if (SHALLOW && !TB && vec_b) {
#pragma unroll
      for (int i = 0; i < NB; ++i)
        load_op(std::integral_constant<bool, !TB>{}, true, B, ldb, n0, N, k0, min(tid / B_VPR + i * B_RPP, K - 1 - k0),
                (tid % B_VPR) * VW, r.b[i]);
    } else {
#pragma unroll
      for (int i = 0; i < NB; ++i)
        load_op(std::integral_constant<bool, !TB>{}, false, B, ldb, n0, N, k0, tid / B_VPR + i * B_RPP,
                (tid % B_VPR) * VW, r.b[i]);
    }
  };
  auto store_slab = [&](auto fast, int buf, int k0, Regs& q) __attribute__((always_inline)) {
    constexpr bool FAST = decltype(fast)::value;
    if (!FAST && k0 + BK > K) {  // the last, partial slab
#pragma unroll
      for (int i = 0; i < NA; ++i)
#pragma unroll
        for (int e = 0; e < VW; ++e)
          if (k0 + (TA ? tid / A_VPR + i * A_RPP : (tid % A_VPR) * VW + e) >= K) q.a[i][e] = T(0);
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int e = 0; e < VW; ++e)
          if (k0 + (TB ? (tid % B_VPR) * VW + e : tid / B_VPR + i * B_RPP) >= K) q.b[i][e] = T(0);
    }
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      const int r = tid / A_VPR + i * A_RPP, c = (tid % A_VPR) * VW;
      if (TA) {  // (k = r, m = c ..) -> As[m][k]
#pragma unroll
        for (int e = 0; e < VW; ++e) As[buf][(c + e) * LDA_S + r] = q.a[i][e];
      } else {
        *reinterpret_cast<VA*>(&As[buf][r * LDA_S + c]) = q.a[i];
      }
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int r = tid / B_VPR + i * B_RPP, c = (tid % B_VPR) * VW;
      if (TB) {  // (n = r, k = c ..) -> Bs[k][n]
#pragma unroll
        for (int e = 0; e < VW; ++e) Bs[buf][(c + e) * LDB_S + r] = q.b[i][e];
      } else {
        *reinterpret_cast<VA*>(&Bs[buf][r * LDB_S + c]) = q.b[i];
      }
    }
  };
  auto multiply_part = [&](auto kend, int buf) __attribute__((always_inline)) {
    const T* as = As[buf];
    const T* bs = Bs[buf];
#pragma unroll
    for (int kk = 0; kk < decltype(kend)::value; kk += 4) {
      T a[FM], b[FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) a[i] = as[(wm0 + i * 16 + lane % 16) * LDA_S + kk + lane / 16];
#pragma unroll
      for (int j = 0; j < FN; ++j) b[j] = bs[(kk + lane / 16) * LDB_S + wn0 + j * 16 + lane % 16];
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = MF::mma(a[i], b[j], acc[i][j]);
    }
  };

  auto multiply = [&](int buf) __attribute__((always_inline)) { multiply_part(std::integral_constant<int, BK>{}, buf); };

  constexpr std::true_type fast{};
  constexpr std::false_type any{};
  const int nk = (K + BK - 1) / BK;
  const int nfast = vec_a && vec_b ? K / BK : 0;  // full slabs, if read by vectors
  Regs ra, rb;
  load_slab(any, 0, ra);
  if (PF == 2 && nk > 1) load_slab(any, BK, rb);
  store_slab(any, 0, 0, ra);
  __syncthreads();
  int kt = 0;
  // A last slab of which at most half lies within K: the other half's products would be zeros (700 x 700,
  // k = 333 FP32: 9.6 us, 10.3 with them; 412 x 346, k = 111 FP64: 5.0, 5.3).  Large tiles are for long K.
  const int half = BM <= 64 && nk * BK - K >= BK / 2;
  if (PF == 1) {
    // Past the end slab 0 is requested again: with the last load left out by a branch 4096^3 FP64
    // takes 2.14 ms instead of 2.02 (and 2.11 as one basic block, where the compiler moves the loads
    // down between the products).
    for (; kt < nk - half; ++kt) {
      load_slab(any, kt + 1 < nk ? (kt + 1) * BK : 0, ra);
      multiply(kt & 1);
      if (kt + 1 < nk) store_slab(any, (kt & 1) ^ 1, (kt + 1) * BK, ra);
      __syncthreads();
    }
  } else {
    // slab kt in LDS buffer kt & 1, slab kt + 1 on its way in the other register set, slab kt + 2
    // requested into the set that held kt.  Full slabs in a loop without branches (2048^3 FP64, both
    // operands transposed: 262 us, 302 with them; 512^3 9.7, 11.7).
    for (; kt + 3 < nfast; kt += 2) {
      load_slab(fast, (kt + 2) * BK, ra);
      multiply(0);
      store_slab(fast, 1, (kt + 1) * BK, rb);
      __syncthreads();
      load_slab(fast, (kt + 3) * BK, rb);
      multiply(1);
      store_slab(fast, 0, (kt + 2) * BK, ra);
      __syncthreads();
    }
    // Past the end slab 0 is requested again: with a conditional load the wait for slab kt + 1 could
    // not leave slab kt + 2 in flight.
    for (; kt < nk - half; kt += 2) {
      load_slab(any, kt + 2 < nk ? (kt + 2) * BK : 0, ra);
      multiply(0);
      if (kt + 1 < nk) store_slab(any, 1, (kt + 1) * BK, rb);
      __syncthreads();
      if (kt + 1 >= nk - half) break;
      load_slab(any, kt + 3 < nk ? (kt + 3) * BK : 0, rb);
      multiply(1);
      if (kt + 2 < nk) store_slab(any, 0, (kt + 2) * BK, ra);
      __syncthreads();
    }
  }
  if (half) multiply_part(std::integral_constant<int, BK / 2>{}, (nk - 1) & 1);

  // Epilogue: C = alpha*acc + beta*C; beta == 0 never reads C (it may hold NaN/garbage).
  const bool read_c = beta != T(0);
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gr = m0 + wm0 + i * 16 + MF::row(r, lane);
        const int gc = n0 + wn0 + j * 16 + lane % 16;
        if (gr < M && gc < N && (!TA || gr >= tm * BM) && (TB || gc >= tn * BN)) {
          T* p = C + (long)gr * ldc + gc;
          T v = alpha * acc[i][j][r];
          if (read_c) v += beta * *p;
          *p = v;
        }
      }
}

template <typename T, int BM, int BN, int WM, int WN, int BK, int PF, bool TA = false, bool TB = false>
__global__ __launch_bounds__(kThreads, 2) void gemm_mfma_kernel(int M, int N, int K, T alpha,
                                                             const T* __restrict__ A, long lda,
                                                             const T* __restrict__ B, long ldb,
                                                             T beta, T* __restrict__ C,
                                                             long ldc) {
  __shared__ GemmShm<T, BM, BN, BK, TA, TB> sh;
  const int tiles_m = (M + BM - 1) / BM;
  const int tiles_n = (N + BN - 1) / BN;
  int tm, tn;
  tile_coords(tiles_m, tiles_n, tm, tn);
  gemm_tile<T, BM, BN, WM, WN, BK, PF, TA, TB>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, tm, tn, sh);
}

// ---- grouped GEMM: many independent products of uneven sizes in one persistent launch ----
// Tile of the grouped kernel: 64 x 64, waves of 32 x 32, one shallow slab ahead.  Its workgroups go from
// tile to tile, four to a CU, so the others' products cover a tile's first loads, and the deeper
// prefetch that a small single product needs costs more than it hides (3000 products of 16..100: 137 us, 171
// with two slabs ahead, 174 with slabs of 32).
constexpr int kGT = 64;
constexpr int kGBK = 16;

// Tiles of one problem; a problem that fails the bzg_dgemm argument rules gets none (and
// status -1 when a status array is given), an empty one none (status 0).
__device__ __forceinline__ int64_t grouped_tiles(const bzg_dgemm_problem& q, int32_t* status) {
  const bool ok = q.m >= 0 && q.n >= 0 && q.k >= 0 && q.m < (1LL << 31) && q.n < (1LL << 31) &&
                  q.k < (1LL << 31) && q.lda >= (q.k > 0 ? q.k : 1) && q.ldb >= (q.n > 0 ? q.n : 1) &&
                  q.ldc >= (q.n > 0 ? q.n : 1) && (q.m == 0 || q.n == 0 || q.C != nullptr) &&
                  (q.m == 0 || q.n == 0 || q.k == 0 || (q.A != nullptr && q.B != nullptr));
  if (status) *status = ok ? 0 : -1;
  if (!ok || q.m == 0 || q.n == 0) return 0;
  return ((q.m + kGT - 1) / kGT) * ((q.n + kGT - 1) / kGT);
}

// prefix[p] = number of 64 x 64 tiles of problems 0..p-1 (p = 0..count); one workgroup.
__global__ __launch_bounds__(1024) void grouped_prefix_kernel(int count, const bzg_dgemm_problem* __restrict__ pr,
                                                              int64_t* __restrict__ prefix,
                                                              int32_t* __restrict__ status) {
  __shared__ int64_t part[1024];
  const int t = threadIdx.x;
  const int per = (count + 1023) / 1024;
  const int b = t * per, e = min(count, b + per);
  int64_t s = 0;
  for (int p = b; p < e; ++p) s += grouped_tiles(pr[p], nullptr);
  part[t] = s;
  __syncthreads();
  if (t == 0) {
    int64_t acc = 0;
    for (int i = 0; i < 1024; ++i) {
      const int64_t v = part[i];
      part[i] = acc;
      acc += v;
    }
  }
  __syncthreads();
  int64_t acc = part[t];
  for (int p = b; p < e; ++p) {
    prefix[p] = acc;
    acc += grouped_tiles(pr[p], status ? status + p : nullptr);
  }
  if (t == 1023) prefix[count] = acc;  // the last range ends at count: acc is the total
}

// Persistent: workgroup w takes tiles w, w + grid, ... of the concatenated tile list (a fixed
// assignment, no atomics); the problem of a tile is found by binary search in the prefix.
// Problems with k == 0 are scaled (C = beta C) tile by tile.
__global__ __launch_bounds__(kThreads, 2) void gemm_grouped_kernel(int count, const bzg_dgemm_problem* __restrict__ pr,
                                                                   const int64_t* __restrict__ prefix) {
  __shared__ GemmShm<double, kGT, kGT, kGBK> sh;
  const int64_t total = prefix[count];
  for (int64_t t = blockIdx.x; t < total; t += gridDim.x) {
    int lo = 0, hi = count - 1;  // last p with prefix[p] <= t
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (prefix[mid] <= t) lo = mid; else hi = mid - 1;
    }
    const bzg_dgemm_problem q = pr[lo];
    const int tiles_n = (int)((q.n + kGT - 1) / kGT);
    const int local = (int)(t - prefix[lo]);
    const int tm = local / tiles_n, tn = local % tiles_n;
    if (q.k == 0) {
      for (int e = threadIdx.x; e < kGT * kGT; e += kThreads) {
        const long r = (long)tm * kGT + e / kGT, c = (long)tn * kGT + e % kGT;
        if (r < q.m && c < q.n) {
          double* p = q.C + r * q.ldc + c;
          *p = (q.beta == 0.0) ? 0.0 : q.beta * *p;
        }
      }
    } else {
      gemm_tile<double, kGT, kGT, 32, 32, kGBK, 1>((int)q.m, (int)q.n, (int)q.k, q.alpha, q.A, q.lda, q.B, q.ldb,
                                                   q.beta, q.C, q.ldc, tm, tn, sh);
    }
    __syncthreads();  // LDS of this tile is free before the next one is staged
  }
}

// C = beta*C for k == 0 (and the empty product).
template <typename T>
__global__ void scale_matrix_kernel(int M, int N, T beta, T* C, long ldc) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (long)M * N) return;
  const long r = idx / N, c = idx % N;
  T* p = C + r * ldc + c;
  *p = (beta == T(0)) ? T(0) : beta * *p;
}

// INT32 GEMM on VALU: 64x64 tile, 256 threads, 4x4 micro-tile per thread.  TA / TB: the
// operand is stored transposed (A as K x M, B as N x K); the staging loop then walks the tile so
// that neighbouring threads read neighbouring addresses.  Wrap-around integer arithmetic is
// exact, so every form gives the same bits as the product of transposed copies.
template <bool TA, bool TB>
__global__ __launch_bounds__(256) void igemm_kernel(int M, int N, int K, uint32_t alpha,
                                                    const int32_t* __restrict__ A, long lda,
                                                    const int32_t* __restrict__ B, long ldb,
                                                    uint32_t beta, int32_t* __restrict__ C,
                                                    long ldc) {
  constexpr int T = 64, BK = 16;
  __shared__ uint32_t As[BK][T + 4];  // transposed: As[k][m]
  __shared__ uint32_t Bs[BK][T + 4];
  const int tid = threadIdx.x;
  const int tiles_n = (N + T - 1) / T;
  const int m0 = (blockIdx.x / tiles_n) * T, n0 = (blockIdx.x % tiles_n) * T;
  const int tr = (tid / 16) * 4, tc = (tid % 16) * 4;
  uint32_t acc[4][4] = {};
  for (int k0 = 0; k0 < K; k0 += BK) {
    for (int e = tid; e < T * BK; e += 256) {
      // A element (m0+r, k0+c): stored at [m][k], or at [k][m] when TA
      const int r = TA ? e % T : e / BK, c = TA ? e / T : e % BK;
      const bool ain = m0 + r < M && k0 + c < K;
      As[c][r] = ain ? (uint32_t)(TA ? A[(long)(k0 + c) * lda + m0 + r] : A[(long)(m0 + r) * lda + k0 + c]) : 0u;
      // B element (k0+kr, n0+nc): stored at [k][n], or at [n][k] when TB
      const int kr = TB ? e % BK : e / T, nc = TB ? e / BK : e % T;
      const bool bin = k0 + kr < K && n0 + nc < N;
      Bs[kr][nc] = bin ? (uint32_t)(TB ? B[(long)(n0 + nc) * ldb + k0 + kr] : B[(long)(k0 + kr) * ldb + n0 + nc]) : 0u;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < BK; ++k) {
      uint32_t a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[k][tr + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = Bs[k][tc + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] += a[i] * b[j];
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int gr = m0 + tr + i, gc = n0 + tc + j;
      if (gr < M && gc < N) {
        int32_t* p = C + (long)gr * ldc + gc;
        uint32_t v = alpha * acc[i][j];
        if (beta != 0u) v += beta * (uint32_t)*p;
        *p = (int32_t)v;
      }
    }
}

template <typename T>
bzg_status check_gemm_args(bzg_context* ctx, int64_t m, int64_t n, int64_t k, const T* A,
                           int64_t lda, const T* B, int64_t ldb, T* C, int64_t ldc, bool ta = false,
                           bool tb = false) {
  BZG_REQUIRE(ctx != nullptr, BZG_ERR_INVALID_ARGUMENT, "gemm: null context");
  BZG_REQUIRE(m >= 0 && n >= 0 && k >= 0, BZG_ERR_INVALID_ARGUMENT, "gemm: negative size");
  BZG_REQUIRE(m < (1LL << 31) && n < (1LL << 31) && k < (1LL << 31), BZG_ERR_UNSUPPORTED,
              "gemm: dimension >= 2^31");
  const int64_t arow = ta ? m : k, brow = tb ? k : n;  // stored row lengths of A and B
  BZG_REQUIRE(lda >= (arow > 0 ? arow : 1) && ldb >= (brow > 0 ? brow : 1) && ldc >= (n > 0 ? n : 1),
              BZG_ERR_INVALID_ARGUMENT, "gemm: leading dimension smaller than row length");
  if (m > 0 && n > 0) BZG_REQUIRE(C != nullptr, BZG_ERR_INVALID_ARGUMENT, "gemm: null C");
  if (m > 0 && n > 0 && k > 0)
    BZG_REQUIRE(A != nullptr && B != nullptr, BZG_ERR_INVALID_ARGUMENT, "gemm: null A or B");
  return BZG_OK;
}

template <typename T, int BM, int BN, int WM, int WN, int BK, int PF, bool TA = false, bool TB = false>
bzg_status launch_tile(bzg_context* ctx, int m, int n, int k, T alpha, const T* A, long lda,
                       const T* B, long ldb, T beta, T* C, long ldc) {
  ProfScope prof(ctx, sizeof(T) == 8 ? "dgemm" : "sgemm");
  const long tiles = (long)((m + BM - 1) / BM) * ((n + BN - 1) / BN);
  BZG_REQUIRE(tiles < (1L << 31), BZG_ERR_UNSUPPORTED, "gemm: too many tiles");
  dim3 grid((unsigned)tiles), block(kThreads);
  hipLaunchKernelGGL((gemm_mfma_kernel<T, BM, BN, WM, WN, BK, PF, TA, TB>), grid, block, 0, ctx->stream, m, n, k, alpha,
                     A, lda, B, ldb, beta, C, ldc);
  BZG_LAUNCH_CHECK();
  return BZG_OK;
}

// ---- tile-shape autotuner ------------------------------------------------------------
// Tile shapes: 0 = 32 x 32, 1 = 64 x 64, 2 = 128 x 128.  bzg_gemm_autotune times the three
// shapes on a product of the given size and records the fastest for that size class
// (ceil(log2) of m, n, k and the element type); later products of the class use it.  All
// shapes give bit-identical results, so tuning changes speed only.
struct TuneKey {
  int type, lm, ln, lk;
  bool operator<(const TuneKey& o) const {
    return std::tie(type, lm, ln, lk) < std::tie(o.type, o.lm, o.ln, o.lk);
  }
};
std::mutex g_tune_mu;
std::map<TuneKey, int> g_tune;

int ceil_log2(int64_t v) {
  int l = 0;
  while ((int64_t(1) << l) < v) ++l;
  return l;
}
TuneKey tune_key(int type, int64_t m, int64_t n, int64_t k) {
  return TuneKey{type, ceil_log2(m), ceil_log2(n), ceil_log2(k)};
}

// Shapes: 0 = 32x32, 1 = 64x64, 2 = 128x128 tiles; 3 = 128x256 (64x128 per wavefront, FP32
// only: its accumulators need 128 registers, 256 in FP64).  131 TFLOP/s at 8192^3 and 4096^3; 128x128, once
// behind, is at 136 and 133 now, which the rule does not use yet.
template <typename T>
constexpr int kShapes = sizeof(T) == 4 ? 4 : 3;
constexpr int kShortK = 4;  // FP32 only, by rule: 64x64 with slabs of 16 and one ahead, as in the grouped kernel

// Tiles against the 256 CUs, from products of 64 .. 8192 rows and columns with k = 20 .. 8192 (us,
// FP64 / FP32).  A large tile reads less per flop but leaves CUs idle in its last round: 128 x 128
// only from 960 tiles and with 92 % of the rounds' slots filled (8192^3: 16.1 ms / 8.1 against 16.9 / 8.5 with
// 64 x 64; 4096^3: 2025 / 1031 against 1993 / 1077; k = 1500, 3700^2, 841 tiles: 749 / 384 against 644 / 356;
// 2936^2, 529 tiles: 615 / 293 against 419 / 232); FP32's 128 x 256 likewise from 480 tiles.  64 x 64 from 600
// tiles (2000^2, k = 1500: 193 / 108 against 248 / 146 with 32 x 32; 1500^2, 576 tiles: 143 / 83 against 141 /
// 83), and from 200 for short k, where the loads ahead of the first product are most of the time (1000^2,
// k = 64: 7.0 / 5.6 against 7.8 / 6.3).  FP32 below k = 64 with shallow slabs, which leave less of the last
// one outside K (1500^2, k = 20: 6.4 us, 8.7 with slabs of 32; 2000^2, k = 48: 9.8, 10.7); at 64 the deep ones
// are ahead (1200^2: 6.6, 6.9).
template <typename T>
int heuristic_shape(int64_t m, int64_t n, int64_t k) {
  auto tiles = [&](int64_t bm, int64_t bn) { return ((m + bm - 1) / bm) * ((n + bn - 1) / bn); };
  auto filled = [](int64_t t) { return t * 100 >= 92 * ((t + 255) / 256 * 256); };
  const int64_t t256 = tiles(128, 256), t128 = tiles(128, 128), t64 = tiles(64, 64);
  if (sizeof(T) == 4 && t256 >= 480 && filled(t256)) return 3;
  if (t128 >= 960 && filled(t128)) return 2;
  if (sizeof(T) == 4 && t64 >= 200 && k < 64) return kShortK;
  if (t64 >= 600 || (t64 >= 200 && k <= (sizeof(T) == 8 ? 128 : 512))) return 1;
  return 0;
}

template <typename T, bool TA = false, bool TB = false>
bzg_status launch_shape_t(bzg_context* ctx, int shape, int64_t m, int64_t n, int64_t k, T alpha, const T* A,
                          int64_t lda, const T* B, int64_t ldb, T beta, T* C, int64_t ldc) {
  if constexpr (sizeof(T) == 4) {
    if (shape == 3)
      return launch_tile<T, 128, 256, 64, 128, 16, 1, TA, TB>(ctx, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
  }
  if constexpr (sizeof(T) == 4) {
    if (shape == kShortK)
      return launch_tile<T, 64, 64, 32, 32, 16, 1, TA, TB>(ctx, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
  }
  if (shape == 2)
    return launch_tile<T, 128, 128, 64, 64, 16, 1, TA, TB>(ctx, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
  if (shape == 1)
    return launch_tile<T, 64, 64, 32, 32, 128 / sizeof(T), 2, TA, TB>(ctx, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
  return launch_tile<T, 32, 32, 16, 16, 256 / sizeof(T), 2, TA, TB>(ctx, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}

template <typename T>
bzg_status launch_shape(bzg_context* ctx, int shape, int64_t m, int64_t n, int64_t k, T alpha, const T* A,
                        int64_t lda, const T* B, int64_t ldb, T beta, T* C, int64_t ldc, bool ta = false,
                        bool tb = false) {
  if (ta && tb) return launch_shape_t<T, true, true>(ctx, shape, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
  if (ta) return launch_shape_t<T, true, false>(ctx, shape, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
  if (tb) return launch_shape_t<T, false, true>(ctx, shape, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
  return launch_shape_t<T, false, false>(ctx, shape, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}

// The longest inner length of one launch: the end of a slab (at most 64) past the last is still an int.
// (Written so in the kernel, without the sum, 412 x 346, k = 111 FP64 takes 5.3 us instead of 5.0.)
constexpr int64_t kMaxK = INT32_MAX - 127;

// Tile choice by size only (never by load), so a product's result never depends on what
// else is running: the tuned shape of the size class if there is one, else heuristic_shape's.
template <typename T>
bzg_status gemm_dispatch(bzg_context* ctx, int64_t m, int64_t n, int64_t k, T alpha, const T* A,
                         int64_t lda, const T* B, int64_t ldb, T beta, T* C, int64_t ldc, bool ta = false,
                         bool tb = false) {
  bzg_status st = check_gemm_args(ctx, m, n, k, A, lda, B, ldb, C, ldc, ta, tb);
  if (st != BZG_OK) return st;
  if (m == 0 || n == 0) return BZG_OK;
  if (k == 0) {
    const long total = m * n;
    hipLaunchKernelGGL(scale_matrix_kernel<T>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                       ctx->stream, (int)m, (int)n, beta, C, (long)ldc);
    BZG_LAUNCH_CHECK();
    return BZG_OK;
  }
  if (k > kMaxK) {
    const int64_t k1 = kMaxK / 2;
    st = gemm_dispatch<T>(ctx, m, n, k1, alpha, A, lda, B, ldb, beta, C, ldc, ta, tb);
    if (st != BZG_OK) return st;
    return gemm_dispatch<T>(ctx, m, n, k - k1, alpha, A + (ta ? k1 * lda : k1), lda, B + (tb ? k1 : k1 * ldb), ldb, T(1),
                            C, ldc, ta, tb);
  }
  int shape = heuristic_shape<T>(m, n, k);
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tune.find(tune_key(sizeof(T) == 8 ? 0 : 1, m, n, k));
    if (it != g_tune.end()) shape = it->second;
  }
  return launch_shape<T>(ctx, shape, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, ta, tb);
}

template <typename T>
bzg_status gemm_autotune(bzg_context* ctx, int64_t m, int64_t n, int64_t k, int32_t* chosen, float* ms_out) {
  BZG_REQUIRE(ctx && m > 0 && n > 0 && k > 0, BZG_ERR_INVALID_ARGUMENT, "gemm_autotune: bad argument");
  BZG_REQUIRE(m < (1LL << 31) && n < (1LL << 31) && k < (1LL << 31), BZG_ERR_UNSUPPORTED,
              "gemm_autotune: dimension >= 2^31");
  k = std::min(k, kMaxK);  // of the same size class
  const size_t bytes = sizeof(T) * ((size_t)m * k + (size_t)k * n + (size_t)m * n);
  void* ws = nullptr;
  bzg_status st = workspace(ctx, 7, bytes, &ws);
  if (st) return st;
  T* A = static_cast<T*>(ws);
  T* B = A + (size_t)m * k;
  T* C = B + (size_t)k * n;
  // operand values do not change the timing of these kernels: zero-filled scratch
  BZG_HIP_CHECK(hipMemsetAsync(ws, 0, bytes, ctx->stream));
  hipEvent_t e0, e1;
  BZG_HIP_CHECK(hipEventCreate(&e0));
  BZG_HIP_CHECK(hipEventCreate(&e1));
  int best = -1;
  float best_ms = 0.f;
  const bool prof = ctx->profile;
  ctx->profile = false;
  for (int shape = 0; shape < kShapes<T> && !st; ++shape) {
    st = launch_shape<T>(ctx, shape, m, n, k, T(1), A, k, B, n, T(0), C, n);  // warm-up
    if (st) break;
    const int reps = 3;
    hipEventRecord(e0, ctx->stream);
    for (int r = 0; r < reps && !st; ++r) st = launch_shape<T>(ctx, shape, m, n, k, T(1), A, k, B, n, T(0), C, n);
    hipEventRecord(e1, ctx->stream);
    if (hipEventSynchronize(e1) != hipSuccess) st = BZG_ERR_HIP;
    float ms = 0.f;
    hipEventElapsedTime(&ms, e0, e1);
    ms /= reps;
    if (!st && (best < 0 || ms < best_ms)) {
      best = shape;
      best_ms = ms;
    }
  }
  ctx->profile = prof;
  hipEventDestroy(e0);
  hipEventDestroy(e1);
  if (st) return st;
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    g_tune[tune_key(sizeof(T) == 8 ? 0 : 1, m, n, k)] = best;
  }
  if (chosen) *chosen = best;
  if (ms_out) *ms_out = best_ms;
  return BZG_OK;
}

}  // namespace
}  // namespace bzg

extern "C" {

bzg_status bzg_dgemm(bzg_context* ctx, int64_t m, int64_t n, int64_t k, double alpha,
                     const double* A, int64_t lda, const double* B, int64_t ldb, double beta,
                     double* C, int64_t ldc) {
  return bzg::gemm_dispatch<double>(ctx, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}

bzg_status bzg_dgemm_grouped(bzg_context* ctx, int64_t count, const bzg_dgemm_problem* problems,
                             int32_t* status) {
  BZG_REQUIRE(ctx != nullptr, BZG_ERR_INVALID_ARGUMENT, "dgemm_grouped: null context");
  BZG_REQUIRE(count >= 0 && count < (1LL << 31), BZG_ERR_INVALID_ARGUMENT, "dgemm_grouped: bad count");
  if (count == 0) return BZG_OK;
  BZG_REQUIRE(problems != nullptr, BZG_ERR_INVALID_ARGUMENT, "dgemm_grouped: null problem array");
  void* ws = nullptr;
  bzg_status st = bzg::workspace(ctx, 6, (size_t)(count + 1) * sizeof(int64_t), &ws);
  if (st) return st;
  int64_t* prefix = static_cast<int64_t*>(ws);
  bzg::ProfScope prof(ctx, "dgemm_grouped");
  hipLaunchKernelGGL(bzg::grouped_prefix_kernel, dim3(1), dim3(1024), 0, ctx->stream, (int)count, problems, prefix,
                     status);
  BZG_LAUNCH_CHECK();
  hipLaunchKernelGGL(bzg::gemm_grouped_kernel, dim3((unsigned)(ctx->num_cus * 4)), dim3(bzg::kThreads), 0,
                     ctx->stream, (int)count, problems, prefix);
  BZG_LAUNCH_CHECK();
  return BZG_OK;
}

bzg_status bzg_gemm_autotune(bzg_context* ctx, int32_t fp32, int64_t m, int64_t n, int64_t k,
                             int32_t* shape, float* ms) {
  return fp32 ? bzg::gemm_autotune<float>(ctx, m, n, k, shape, ms)
              : bzg::gemm_autotune<double>(ctx, m, n, k, shape, ms);
}

bzg_status bzg_gemm_tuning_clear(void) {
  std::lock_guard<std::mutex> lk(bzg::g_tune_mu);
  bzg::g_tune.clear();
  return BZG_OK;
}

bzg_status bzg_sgemm(bzg_context* ctx, int64_t m, int64_t n, int64_t k, float alpha,
                     const float* A, int64_t lda, const float* B, int64_t ldb, float beta,
                     float* C, int64_t ldc) {
  return bzg::gemm_dispatch<float>(ctx, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}

bzg_status bzg_dgemm_ex(bzg_context* ctx, int32_t transa, int32_t transb, int64_t m, int64_t n, int64_t k,
                        double alpha, const double* A, int64_t lda, const double* B, int64_t ldb, double beta,
                        double* C, int64_t ldc) {
  return bzg::gemm_dispatch<double>(ctx, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, transa != 0, transb != 0);
}

bzg_status bzg_sgemm_ex(bzg_context* ctx, int32_t transa, int32_t transb, int64_t m, int64_t n, int64_t k,
                        float alpha, const float* A, int64_t lda, const float* B, int64_t ldb, float beta,
                        float* C, int64_t ldc) {
  return bzg::gemm_dispatch<float>(ctx, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, transa != 0, transb != 0);
}

bzg_status bzg_igemm_ex(bzg_context* ctx, int32_t transa, int32_t transb, int64_t m, int64_t n, int64_t k,
                        int32_t alpha, const int32_t* A, int64_t lda, const int32_t* B, int64_t ldb,
                        int32_t beta, int32_t* C, int64_t ldc) {
  const bool ta = transa != 0, tb = transb != 0;
  bzg_status st = bzg::check_gemm_args(ctx, m, n, k, A, lda, B, ldb, C, ldc, ta, tb);
  if (st != BZG_OK) return st;
  if (m == 0 || n == 0) return BZG_OK;
  {
    // the INT8 matrix cores where they measured faster than the vector ALUs (MI355X: from
    // 256 x 256 x 4096 up, 2.7x at 1024^3, 4.5x at 8192^3; even at 1024 x 1024 x 256): k >= 512
    // and at least one 256 x 256 tile of output, or k >= 256 and 2048 x 2048; m and n >= 128
    // (the digit GEMM pads both to 256: skinny products stay on the VALU); a digit workspace
    // of at most 8 GiB (one K chunk of the digits and the 4 class planes)
    const int64_t mp = (m + 255) / 256 * 256, np = (n + 255) / 256 * 256;
    const int64_t kp = std::min<int64_t>((k + 127) / 128 * 128, bzg::kIgemmDigitsChunk);
    const double ws_bytes = 16.0 * mp * np + 4.0 * (mp + np) * kp;
    const double mn = (double)m * (double)n;
    if (((k >= 512 && mn >= 65536.0) || (k >= 256 && mn >= 4194304.0)) && std::min(m, n) >= 128 &&
        ws_bytes <= 8.0 * (1L << 30))
      return bzg::igemm_digits_impl(ctx, ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
  }
  const long tiles = ((m + 63) / 64) * ((n + 63) / 64);
  BZG_REQUIRE(tiles < (1L << 31), BZG_ERR_UNSUPPORTED, "igemm: too many tiles");
  const dim3 grid((unsigned)tiles), block(256);
#define BZG_IGEMM(TA_, TB_)                                                                                  \
  hipLaunchKernelGGL((bzg::igemm_kernel<TA_, TB_>), grid, block, 0, ctx->stream, (int)m, (int)n, (int)k,   \
                     (uint32_t)alpha, A, (long)lda, B, (long)ldb, (uint32_t)beta, C, (long)ldc)
  if (ta && tb) BZG_IGEMM(true, true);
  else if (ta) BZG_IGEMM(true, false);
  else if (tb) BZG_IGEMM(false, true);
  else BZG_IGEMM(false, false);
#undef BZG_IGEMM
  BZG_LAUNCH_CHECK();
  return BZG_OK;
}

bzg_status bzg_igemm_digits(bzg_context* ctx, int32_t transa, int32_t transb, int64_t m, int64_t n, int64_t k,
                            int32_t alpha, const int32_t* A, int64_t lda, const int32_t* B, int64_t ldb,
                            int32_t beta, int32_t* C, int64_t ldc) {
  const bool ta = transa != 0, tb = transb != 0;
  bzg_status st = bzg::check_gemm_args(ctx, m, n, k, A, lda, B, ldb, C, ldc, ta, tb);
  if (st != BZG_OK) return st;
  if (m == 0 || n == 0) return BZG_OK;
  if (k == 0) return bzg_igemm_ex(ctx, transa, transb, m, n, 0, alpha, A, lda, B, ldb, beta, C, ldc);
  return bzg::igemm_digits_impl(ctx, ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}

bzg_status bzg_igemm(bzg_context* ctx, int64_t m, int64_t n, int64_t k, int32_t alpha,
                     const int32_t* A, int64_t lda, const int32_t* B, int64_t ldb,
                     int32_t beta, int32_t* C, int64_t ldc) {
  return bzg_igemm_ex(ctx, 0, 0, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}

}  // extern "C"
