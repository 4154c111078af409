// K2/K3: right-looking blocked LU with partial pivoting (FP64 and FP32) for
// row-major matrices on gfx950.
//
// Replaces the factorisations that the reference runs through XLA/LAPACK:
// jnp.linalg.inv (updes/assembly.py:90, getrf + getri) and lineax QR
// (updes/operators.py:612-613).  The augmented collocation matrix is factored
// once: P K = L U.
//
// Structure per outer panel of NB columns (k0 .. k0+NB):
//   1. panel factorisation, leaf by leaf (64 columns): a leaf runs as ONE
//      launch of co-resident workgroups that keep their rows of the leaf in
//      registers and agree on every pivot through one exchange per column
//      (every workgroup publishes its best row and a tagged record, all of
//      them poll the records and pick the same winner); a second launch
//      applies its interchanges to the panel's other columns and solves for
//      U12 of its rows, and one product updates what is right and below.  The
//      inverse of the panel's unit-lower block grows by a row block per leaf,
//      beside the next one; its last block and the plan of the panel's
//      interchanges are one launch.  (FP64 systems of up to kRecursiveRows
//      rows: by recursive halving, whose splits solve and join inverses with
//      products.)
//   2. row interchanges of the columns outside the panel through a
//      gather/scatter plan (row-major rows are contiguous, so a swap is a
//      coalesced copy);
//   3. U12 = inv(L11) A12 with the MFMA GEMM;
//   4. trailing update A22 -= L21 U12 with an MFMA GEMM
//      (v_mfma_f64_16x16x4f64 / v_mfma_f32_16x16x4f32, 128x128 tiles,
//      k-tiles loaded global -> LDS by DMA, XCD-aware tile order).
#include <algorithm>
#include <atomic>
#include <mutex>
#include <type_traits>
#include <vector>

#include "common.h"

namespace rbfx {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

template <typename T>
struct Mma;
// MFMA 16x16x4 operand layout (both types): lane l holds A[l%16][l/16] and
// B[l/16][l%16].  Accumulator element v of lane l is D[row(l,v)][l%16] with
//   f32: row = 4*(l/16) + v        f64: row = 4*v + l/16
// (measured on gfx950 with one-hot operands).
template <>
struct Mma<double> {
  typedef v4d acc_t;
  static constexpr int BK = 8;
  __device__ static inline acc_t mma(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  __device__ static inline int row(int lane, int v) { return 4 * v + (lane >> 4); }
};
template <>
struct Mma<float> {
  typedef v4f acc_t;
  static constexpr int BK = 16;
  __device__ static inline acc_t mma(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  __device__ static inline int row(int lane, int v) { return 4 * (lane >> 4) + v; }
};

// ---------------------------------------------------------------------------
// GEMM: C = beta*C + alpha*A*B, row-major, beta in {0,1}.
// Block tile 128x128, 4 waves (2x2), wave tile 64x64 = 4x4 MFMA 16x16 tiles.
constexpr int GBM = 128, GBN = 128, GTHREADS = 256;

// Register-staged version: the k-tiles of A and B are loaded two tiles
// ahead into two register slots and stored to an LDS double buffer.  It
// serves the shapes and alpha values the LDS-DMA kernel below does not take.
// Two waves per SIMD (<= 256 registers each) so one wave's barrier or load
// wait overlaps the other's MFMAs.
// USE only separates the kernel symbols of the trailing update (0), of the
// triangular solve (1), of the diagonal-block inverse (2) and of the updates
// inside a recursive panel (3) in profiles; the code is the same.
template <typename T, int USE>
__global__ __launch_bounds__(GTHREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_kernel(
                                                        int64_t m, int64_t n, int64_t k, T alpha,
                                                        const T* __restrict__ A, int64_t lda,
                                                        const T* __restrict__ B, int64_t ldb,
                                                        T beta, T* __restrict__ C, int64_t ldc,
                                                        int64_t tiles_m, int64_t tiles_n) {
  constexpr int BK = Mma<T>::BK;
  constexpr int AV = GBM * BK / GTHREADS;  // A elements per thread per k-tile
  constexpr int BV = BK * GBN / GTHREADS;  // B elements per thread per k-tile
  // double-buffered k-tiles: the next tile is written while this one is read
  __shared__ T As[2][BK][GBM];
  __shared__ T Bs[2][BK][GBN];

  // Tile order.  Tiles are numbered in groups of 8 tile rows, column by
  // column inside a group, so the ~64 workgroups resident on one XCD at a
  // time cover an 8 x 8 patch and share its A and B tiles in that XCD's L2.
  // Consecutive workgroup ids land on different XCDs (round robin), so XCD x
  // takes the x-th contiguous eighth of that numbering.
  const int64_t T_ = tiles_m * tiles_n;
  const int64_t L = blockIdx.x;
  const int64_t per = (T_ + 7) / 8;
  const int64_t tile = (L % 8) * per + L / 8;
  if (tile >= T_) return;
  constexpr int64_t kGroupM = 8;
  const int64_t gwidth = kGroupM * tiles_n;
  const int64_t first_m = (tile / gwidth) * kGroupM;
  const int64_t gm = tiles_m - first_m < kGroupM ? tiles_m - first_m : kGroupM;
  const int64_t tm = first_m + (tile % gwidth) % gm;
  const int64_t tn = (tile % gwidth) / gm;
  const int64_t row0 = tm * GBM, col0 = tn * GBN;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wid = tid >> 6;
  const int wm = wid >> 1, wn = wid & 1;

  // The accumulators start from beta*C (beta is 0 or 1) and alpha is folded
  // into the A tile, so the epilogue only stores (no C reads held live).
  typename Mma<T>::acc_t acc[4][4];
  const bool add = beta != T(0);
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t c = col0 + wn * 64 + j * 16 + (lane & 15);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t r = row0 + wm * 64 + i * 16 + Mma<T>::row(lane, v);
        acc[i][j][v] = (add && r < m && c < n) ? C[r * ldc + c] : T(0);
      }
    }

  // global -> register staging maps
  // A tile (GBM x BK): thread -> row ar = tid % GBM, k chunk ak = (tid / GBM) * AV
  const int ar = tid % GBM, ak = (tid / GBM) * AV;
  // B tile (BK x GBN): thread -> k row bk = tid / (GBN / BV), col chunk bc
  const int bk = tid / (GBN / BV), bc = (tid % (GBN / BV)) * BV;
  // Two register slots: the loads of k-tile t+2 are issued while tile t is
  // multiplied, so a load has two tiles of MFMA work to arrive.
  T ra0[AV], rb0[BV], ra1[AV], rb1[BV];

  auto load = [&](int64_t kt, T (&ra)[AV], T (&rb)[BV]) {
    const int64_t gr = row0 + ar;
    const int64_t gk = kt + ak;
    const T* pa = A + gr * lda + gk;
    if (gr < m && gk + AV <= k) {
#pragma unroll
      for (int q = 0; q < AV; ++q) ra[q] = pa[q];
    } else {
#pragma unroll
      for (int q = 0; q < AV; ++q) ra[q] = (gr < m && gk + q < k) ? pa[q] : T(0);
    }
    const int64_t gkb = kt + bk;
    const int64_t gc = col0 + bc;
    const T* pb = B + gkb * ldb + gc;
    if (gkb < k && gc + BV <= n) {
#pragma unroll
      for (int q = 0; q < BV; ++q) rb[q] = pb[q];
    } else {
#pragma unroll
      for (int q = 0; q < BV; ++q) rb[q] = (gkb < k && gc + q < n) ? pb[q] : T(0);
    }
  };
  auto store = [&](int buf, const T (&ra)[AV], const T (&rb)[BV]) {
#pragma unroll
    for (int q = 0; q < AV; ++q) As[buf][ak + q][ar] = alpha * ra[q];
#pragma unroll
    for (int q = 0; q < BV; ++q) Bs[buf][bk][bc + q] = rb[q];
  };
  auto compute = [&](int buf) {
#pragma unroll
    for (int kk = 0; kk < BK; kk += 4) {
      T af[4], bf[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) af[i] = As[buf][kk + (lane >> 4)][wm * 64 + i * 16 + (lane & 15)];
#pragma unroll
      for (int j = 0; j < 4; ++j) bf[j] = Bs[buf][kk + (lane >> 4)][wn * 64 + j * 16 + (lane & 15)];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = Mma<T>::mma(af[i], bf[j], acc[i][j]);
    }
  };

  load(0, ra0, rb0);
  if (BK < k) load(BK, ra1, rb1);
  store(0, ra0, rb0);
  __syncthreads();
  // LDS buffer 0 holds the even k-tiles, buffer 1 the odd ones; slot 0 the
  // register copy of the next even tile, slot 1 of the next odd one.  A
  // buffer is rewritten only after the barrier that follows its last reads.
  for (int64_t kt = 0; kt < k; kt += 2 * BK) {
    if (kt + 2 * BK < k) load(kt + 2 * BK, ra0, rb0);
    compute(0);
    if (kt + BK < k) store(1, ra1, rb1);
    __syncthreads();
    if (kt + BK >= k) break;
    if (kt + 3 * BK < k) load(kt + 3 * BK, ra1, rb1);
    compute(1);
    if (kt + 2 * BK < k) store(0, ra0, rb0);
    __syncthreads();
  }

  // epilogue: plain stores
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t c = col0 + wn * 64 + j * 16 + (lane & 15);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t r = row0 + wm * 64 + i * 16 + Mma<T>::row(lane, v);
        if (r < m && c < n) C[r * ldc + c] = acc[i][j][v];
      }
    }
  }
}

// GEMM with LDS-DMA operand loads (global_load_lds_dwordx4): the k-tiles go
// from global memory straight into a ring of kGemmStages LDS stages, so no
// registers stage them and a tile is requested kGemmStages-1 tiles before it
// is multiplied.  One barrier per k-tile.
//
// Layouts (E = 16 / sizeof(T) elements per 16-byte chunk):
//   A stage: 128 rows x BK, chunk (m, g) = A[m][E g .. E g + E) at position
//     4 m + (g ^ ((m >> 2) & 3))  (the xor keeps the 16-lane groups of the
//     operand reads on distinct banks);
//   B stage: BK rows x 128, chunk (k, q) = B[k][E q .. E q + E) at k*(128/E) + q.
// MFMA k-assignment: lane group g = lane/16 of MFMA s (0 <= s < E) holds
// k = E g + s, so one 16-byte read gives a lane its A values of all E MFMAs.
// For B one 16-byte read gives E adjacent columns, which feed E adjacent
// n-tiles: tile j's column for lane column c is 16E (j/E) + E c + j%E.
// Requirements (checked by the host): k % BK == 0, lda, ldb and ldc multiples
// of E, 16-byte aligned A, B and C, and rows of B and C that hold the whole
// last chunk (ld >= n rounded up to E): its columns past n are read, and only
// those before n are stored.
constexpr int kGemmStages = 4;

// BT x BT block tile (BT = 128, or 64 for small FP64 products), 2 x 2 waves
// of (BT/2) x (BT/2), each TW x TW MFMA 16x16 tiles.
template <typename T, int USE, int BT, int STAGES = kGemmStages>
__device__ __forceinline__ void gemm_dma_body(int64_t m, int64_t n, int64_t k, T alpha, const T* __restrict__ A,
                                              int64_t lda, const T* __restrict__ B, int64_t ldb, T beta,
                                              T* __restrict__ C, int64_t ldc, int64_t tiles_m, int64_t tiles_n) {
  constexpr int BK = Mma<T>::BK;
  constexpr int E = 16 / (int)sizeof(T);
  constexpr int TW = BT / 32;      // MFMA tiles per wave and dimension
  constexpr int HB = BT / 2;       // wave tile extent
  constexpr int NG = BT / E;       // chunks per B row
  constexpr int NCH = 4 * BT;      // chunks per operand and stage
  constexpr int RC = NCH / GTHREADS;  // chunks per thread and operand
  static_assert(4 * E == BK, "one 16-byte chunk per lane group and k-tile");
  static_assert(BT * (BK / E) == NCH && BK * NG == NCH, "chunk counts");
  static_assert(TW % E == 0 || E == 2, "E adjacent n-tiles per 16-byte B read");
  static_assert(TW >= E, "E adjacent n-tiles per 16-byte B read");
  typedef T vec_t __attribute__((ext_vector_type(E)));
  __shared__ __align__(16) T sm[STAGES][2][NCH * E];

  // tile order as in gemm_kernel (groups of 8 tile rows, XCD-contiguous)
  const int64_t T_ = tiles_m * tiles_n;
  const int64_t L = blockIdx.x;
  const int64_t per = (T_ + 7) / 8;
  const int64_t tile = (L % 8) * per + L / 8;
  if (tile >= T_) return;
  constexpr int64_t kGroupM = 8;
  const int64_t gwidth = kGroupM * tiles_n;
  const int64_t first_m = (tile / gwidth) * kGroupM;
  const int64_t gm = tiles_m - first_m < kGroupM ? tiles_m - first_m : kGroupM;
  const int64_t tm = first_m + (tile % gwidth) % gm;
  const int64_t tn = (tile % gwidth) / gm;
  const int64_t row0 = tm * BT, col0 = tn * BT;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wid = tid >> 6;
  const int wm = wid >> 1, wn = wid & 1;
  const int lg = lane >> 4, lc = lane & 15;

  // DMA sources of this thread (RC A chunks, RC B chunks per k-tile); rows
  // past m and chunks past n are clamped (their results are never stored)
  const T* srcA[RC];
  const T* srcB[RC];
#pragma unroll
  for (int r = 0; r < RC; ++r) {
    const int p = (r * 4 + wid) * 64 + lane;
    const int mm = p >> 2, g = (p & 3) ^ ((mm >> 2) & 3);
    const int64_t row = row0 + mm < m ? row0 + mm : m - 1;
    srcA[r] = A + row * lda + g * E;
    const int kk = p / NG, q = p % NG;
    const int64_t col = col0 + (int64_t)q * E < n ? col0 + (int64_t)q * E : (n - 1) / E * E;
    srcB[r] = B + (int64_t)kk * ldb + col;
  }
  auto issue = [&](int64_t kt, int st) {
#pragma unroll
    for (int r = 0; r < RC; ++r) {
      const int base = (r * 4 + wid) * 64 * E;
      __builtin_amdgcn_global_load_lds((const void*)(srcA[r] + kt),
                                       (__attribute__((address_space(3))) void*)(&sm[st][0][base]), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((const void*)(srcB[r] + kt * ldb),
                                       (__attribute__((address_space(3))) void*)(&sm[st][1][base]), 16, 0, 0);
    }
  };

  typename Mma<T>::acc_t acc[TW][TW];
  const bool add = beta != T(0);
  // alpha is +-1 here: the sum runs on alpha*C and alpha is applied at the end
  const bool neg = alpha < T(0);
#pragma unroll
  for (int i = 0; i < TW; ++i)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int64_t r = row0 + wm * HB + i * 16 + Mma<T>::row(lane, v);
#pragma unroll
      for (int jg = 0; jg < TW / E; ++jg) {
        const int64_t c = col0 + wn * HB + 16 * E * jg + E * lc;
        vec_t x = {};
        if (add && r < m && c < n) x = *reinterpret_cast<const vec_t*>(C + r * ldc + c);
#pragma unroll
        for (int e = 0; e < E; ++e) acc[i][jg * E + e][v] = neg ? -x[e] : x[e];
      }
    }

  const int64_t nt = k / BK;
#pragma unroll
  for (int t = 0; t < STAGES - 1; ++t)
    if (t < nt) issue((int64_t)t * BK, t);

  for (int64_t t = 0; t < nt; ++t) {
    // tile t has landed once at most (tiles issued after it) x 2 RC loads of
    // this thread are outstanding; the barrier makes every thread's part
    // visible and ends all reads of the stage refilled below
    const int64_t ahead = nt - 1 - t < STAGES - 2 ? nt - 1 - t : STAGES - 2;
    if (ahead >= 2)
      __builtin_amdgcn_s_waitcnt(0xF70 | (4 * RC));
    else if (ahead == 1)
      __builtin_amdgcn_s_waitcnt(0xF70 | (2 * RC));
    else
      __builtin_amdgcn_s_waitcnt(0xF70);
    // A plain barrier: __syncthreads() would also wait for the loads of the
    // tiles still in flight (its release fence covers the LDS-DMA).  Every
    // LDS read of this wave has completed (the MFMAs consumed them).
    __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (t + STAGES - 1 < nt) issue((t + STAGES - 1) * BK, (int)((t + STAGES - 1) % STAGES));
    const int st = (int)(t % STAGES);
    const T* As = sm[st][0];
    const T* Bs = sm[st][1];
    vec_t a[TW], b[TW / E][E];
#pragma unroll
    for (int i = 0; i < TW; ++i) {
      const int mm = wm * HB + i * 16 + lc;
      a[i] = *reinterpret_cast<const vec_t*>(As + (mm * 4 + (lg ^ ((mm >> 2) & 3))) * E);
    }
#pragma unroll
    for (int jg = 0; jg < TW / E; ++jg)
#pragma unroll
      for (int s2 = 0; s2 < E; ++s2)
        b[jg][s2] = *reinterpret_cast<const vec_t*>(Bs + ((E * lg + s2) * NG + wn * HB / E + 16 * jg + lc) * E);
#pragma unroll
    for (int s2 = 0; s2 < E; ++s2)
#pragma unroll
      for (int i = 0; i < TW; ++i)
#pragma unroll
        for (int j = 0; j < TW; ++j) acc[i][j] = Mma<T>::mma(a[i][s2], b[j / E][s2][j % E], acc[i][j]);
  }

#pragma unroll
  for (int i = 0; i < TW; ++i)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int64_t r = row0 + wm * HB + i * 16 + Mma<T>::row(lane, v);
      if (r >= m) continue;
#pragma unroll
      for (int jg = 0; jg < TW / E; ++jg) {
        const int64_t c = col0 + wn * HB + 16 * E * jg + E * lc;
        if (c >= n) continue;
        vec_t x;
#pragma unroll
        for (int e = 0; e < E; ++e) x[e] = neg ? -acc[i][jg * E + e][v] : acc[i][jg * E + e][v];
        if (c + E <= n) {
          *reinterpret_cast<vec_t*>(C + r * ldc + c) = x;
        } else {
          for (int e = 0; c + e < n; ++e) C[r * ldc + c + e] = x[e];
        }
      }
    }
}

template <typename T, int USE, int STAGES = kGemmStages>
__global__ __launch_bounds__(GTHREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_dma_kernel(
    int64_t m, int64_t n, int64_t k, T alpha, const T* __restrict__ A, int64_t lda, const T* __restrict__ B,
    int64_t ldb, T beta, T* __restrict__ C, int64_t ldc, int64_t tiles_m, int64_t tiles_n) {
  gemm_dma_body<T, USE, 128, STAGES>(m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, tiles_m, tiles_n);
}

// 64 x 64 tiles for FP64 products too small to fill the GPU with 128 x 128
// tiles (the in-panel updates, inverses and triangular solves of late
// panels): four times the workgroups, a quarter of the k-loop work each.
template <int USE>
__global__ __launch_bounds__(GTHREADS) void gemm_dma64_kernel(int64_t m, int64_t n, int64_t k, double alpha,
                                                             const double* __restrict__ A, int64_t lda,
                                                             const double* __restrict__ B, int64_t ldb,
                                                             double beta, double* __restrict__ C, int64_t ldc,
                                                             int64_t tiles_m, int64_t tiles_n) {
  gemm_dma_body<double, USE, 64>(m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, tiles_m, tiles_n);
}

// small_lds: an FP32 product of the panel stream, which runs beside the
// trailing update: a two-stage ring (32 KB of LDS), so that its workgroups
// fit beside two update workgroups on a CU instead of waiting for one to end.
template <typename T, int USE = 0>
static int gemm_launch(int64_t m, int64_t n, int64_t k, T alpha, const T* A, int64_t lda, const T* B,
                       int64_t ldb, T beta, T* C, int64_t ldc, hipStream_t s, bool small_lds = false,
                       bool ragged = true) {
  if (m <= 0 || n <= 0) return RBFX_OK;
  const int64_t tm = ceil_div(m, GBM), tn = ceil_div(n, GBN);
  const int64_t tiles = tm * tn;
  const int64_t grid = ((tiles + 7) / 8) * 8;
  constexpr int E = 16 / (int)sizeof(T);
  auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  const bool dma = (alpha == T(1) || alpha == T(-1)) && k > 0 && k % Mma<T>::BK == 0 && (n % E == 0 || ragged) && n >= E &&
                   ldb >= ceil_div(n, (int64_t)E) * E &&
                   ldc >= ceil_div(n, (int64_t)E) * E && lda % E == 0 && ldb % E == 0 &&
                   ldc % E == 0 && al16(A) && al16(B) && al16(C);
  if (dma && sizeof(T) == 8 && tiles < 2 * (int64_t)device_info().num_cus) {
    const int64_t tm64 = ceil_div(m, (int64_t)64), tn64 = ceil_div(n, (int64_t)64);
    const int64_t grid64 = ((tm64 * tn64 + 7) / 8) * 8;
    hipLaunchKernelGGL((gemm_dma64_kernel<USE>), dim3((unsigned)grid64), dim3(GTHREADS), 0, s, m, n, k,
                       (double)alpha, reinterpret_cast<const double*>(A), lda, reinterpret_cast<const double*>(B),
                       ldb, (double)beta, reinterpret_cast<double*>(C), ldc, tm64, tn64);
  } else if (dma && small_lds && sizeof(T) == 4)
    hipLaunchKernelGGL((gemm_dma_kernel<T, USE, 2>), dim3((unsigned)grid), dim3(GTHREADS), 0, s, m, n, k, alpha, A,
                       lda, B, ldb, beta, C, ldc, tm, tn);
  else if (dma)
    hipLaunchKernelGGL((gemm_dma_kernel<T, USE>), dim3((unsigned)grid), dim3(GTHREADS), 0, s, m, n, k, alpha, A,
                       lda, B, ldb, beta, C, ldc, tm, tn);
  else
    hipLaunchKernelGGL((gemm_kernel<T, USE>), dim3((unsigned)grid), dim3(GTHREADS), 0, s, m, n, k, alpha, A,
                       lda, B, ldb, beta, C, ldc, tm, tn);
  RBFX_CHECK_LAUNCH();
  return RBFX_OK;
}

template <typename T>
static int gemm(int64_t m, int64_t n, int64_t k, T alpha, const T* A, int64_t lda, const T* B,
                int64_t ldb, T beta, T* C, int64_t ldc, hipStream_t s, bool in_panel = false, bool ragged = true) {
  if (m <= 0 || n <= 0) return RBFX_OK;
  // profile names: the trailing update of the factorisation (and direct
  // calls) vs the updates inside a recursive panel
  const int pid = prof_start(in_panel ? (sizeof(T) == 8 ? "gemm_panel_f64" : "gemm_panel_f32")
                                      : (sizeof(T) == 8 ? "gemm_f64" : "gemm_f32"),
                             s);
  const int st = in_panel ? gemm_launch<T, 3>(m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, s, true, ragged)
                          : gemm_launch<T, 0>(m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, s, false, ragged);
  prof_stop(pid, s, 2.0 * m * n * k, (double)sizeof(T) * (2.0 * m * n + (double)m * k + (double)k * n));
  return st;
}


// Row block b (64 rows, the last one w) of the inverse X of an outer panel's
// unit-lower diagonal block: X_b0 .. X_bb from the rows of L and X above.
template <typename T>
struct InvArgs {
  const T* P = nullptr;  // first row and column of the outer panel
  int64_t lda = 0;
  T* X = nullptr;
  int64_t ldx = 0;
  int b = -1, w = 0;
};

template <typename T>
struct PanelArgs {
  T* A;           // panel top-left (absolute row r0, column r0)
  int64_t lda;
  int64_t m;      // rows in the panel (r0 .. r0+m)
  int w;          // panel width <= kPanelWMax
  int64_t R;      // rows per workgroup
  int64_t r0;     // absolute row of the panel's first row
  int G;          // workgroups of the leaf; the ones past it invert (below)
  int* moves;     // [kMoveStride] out: the leaf's winners, final positions of its first rows, o and w
  int o;          // first column of the leaf in its outer panel
  InvArgs<T> inv; // a finished diagonal block whose rows of the panel's inverse ride along
  int64_t* ipiv;  // (w) absolute pivot rows
  double* cand;   // [2][G][kRecWords] tagged (|value|, row) records (first two words used)
  unsigned long long* cand_row;  // [2][G][kRowStride<T>] tagged words of the candidate rows
  unsigned seq_base;  // step count before this launch
  int* status;
  int32_t* info;
  uint64_t wait_ticks;  // real-time bound of each wait (wall_clock64 ticks)
};

constexpr int kPanelThreads = 256;     // leaf workgroups that run beside a trailing update
constexpr int kPanelWMax = 64;
constexpr int kMoveStride = 2 * kPanelWMax + 2;
// A published row entry carries its own tag: each 64-bit word holds 32 bits
// of the value and the 32-bit tag of its column, so a reader that finds the
// tag has the value, and the writer need not wait between the row and the
// record that announces it.
template <typename T>
constexpr int kRowWords = sizeof(T) / 4;
// a published row: kPanelWMax entries and the reciprocal of the first
template <typename T>
constexpr int kRowStride = (kPanelWMax + 2) * kRowWords<T>;
// Narrow leaves, on request only (rbfx_set_narrow_leaf_rows): a 16-wide FP64
// leaf (72 VGPRs) displaces less of the trailing update than a 64-wide one
// (246).  It paid when a panel cost more than the update beside it and two
// update workgroups left it room (2 x 216 of 512, now 2 x 224); now an FP64 LU
// takes 832 ms with them and 835 ms without at n = 40,006, 466 and 464 ms at
// n = 32,006.
constexpr int kPanelWNarrow = 16;
static std::atomic<int64_t> g_narrow_leaf_rows{0};
// A pivot record (two 64-bit words) owns a 128-byte line: every workgroup
// polls every record, and records sharing a line would serialise the polls.
constexpr int kRecWords = 16;

// Pivot keys.  A candidate (|value|, row) is compared as one 64-bit key:
// the bits of |value| with the low kKeyLow bits replaced by the position of
// the row, inverted so that a lower position wins a tie of the truncated
// values:  bits 11..19 = 511 - workgroup, bits 0..10 = 2047 - row within the
// workgroup.  |value| >= 0, so its bits order like the values; key 0 means
// "no candidate" (no active row, or NaN).  The choice is partial pivoting on
// values rounded down to 32 mantissa bits, ties to the lowest row.
constexpr int kKeyLow = 20;
constexpr unsigned long long kKeyValMask = ~((1ull << kKeyLow) - 1);
constexpr int kKeyMaxGroups = 512, kKeyMaxRows = 2048;
constexpr unsigned long long kKeyBad = ~0ull;  // not a key (a NaN value): the exchange failed

__device__ inline unsigned long long pivot_key(double absval, int q, int local) {
  if (!(absval >= 0.0)) return 0ull;
  return ((unsigned long long)__double_as_longlong(absval) & kKeyValMask) |
         ((unsigned long long)(kKeyMaxGroups - 1 - q) << 11) | (unsigned long long)(kKeyMaxRows - 1 - local);
}

// Maximum of an unsigned value over lanes 0 .. 16 STEP_ROWS of the wave with
// DPP row shifts and broadcasts (no LDS traffic): an inclusive max-scan
// inside each row of 16 lanes, then row 15 -> rows 1, 3 and lane 31 -> rows
// 2, 3, so lane 63 (lane 15 of a single row) holds the result.
template <int CTRL, int ROWMASK>
__device__ inline unsigned dpp_max(unsigned v) {
  const unsigned o = (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWMASK, 0xf, false);
  return v > o ? v : o;
}
template <int LANES>
__device__ inline unsigned wave_max_u32(unsigned v) {
  static_assert(LANES == 16 || LANES == 64, "one row or the whole wave");
  v = dpp_max<0x111, 0xf>(v);  // row_shr:1
  v = dpp_max<0x112, 0xf>(v);  // row_shr:2
  v = dpp_max<0x114, 0xf>(v);  // row_shr:4
  v = dpp_max<0x118, 0xf>(v);  // row_shr:8
  if constexpr (LANES == 64) {
    v = dpp_max<0x142, 0xa>(v);  // row_bcast:15
    v = dpp_max<0x143, 0xc>(v);  // row_bcast:31
  }
  return (unsigned)__builtin_amdgcn_readlane((int)v, LANES - 1);
}
__device__ inline unsigned long long umax64(unsigned long long a, unsigned long long b) { return a > b ? a : b; }
// Maximum of a 64-bit key: the high words first (one 32-bit step per DPP
// move), then the low words of the lanes that hold that maximum, usually one.
template <int LANES = 64>
__device__ inline unsigned long long wave_max_key(unsigned long long v) {
  const unsigned hi = (unsigned)(v >> 32), lo = (unsigned)v;
  const unsigned mh = wave_max_u32<LANES>(hi);
  const unsigned long long top = __ballot(hi == mh && (LANES == 64 || (threadIdx.x & 63) < LANES));
  unsigned ml;
  if ((top & (top - 1)) == 0)
    ml = (unsigned)__builtin_amdgcn_readlane((int)lo, __ffsll((long long)top) - 1);
  else
    ml = wave_max_u32<LANES>(hi == mh ? lo : 0u);
  return ((unsigned long long)mh << 32) | ml;
}

// Block-wide key maximum; one barrier.  s has one slot per wave and is
// reused by a later call only after at least one more barrier.
template <int NT>
__device__ inline unsigned long long block_max_key(unsigned long long key, unsigned long long* s) {
  constexpr int NW = NT / 64;
  const unsigned long long wm = wave_max_key(key);
  const int lane = threadIdx.x & 63;
  if (lane == 0) s[threadIdx.x >> 6] = wm;
  __syncthreads();
  if constexpr (NW <= 4) {
    unsigned long long b = s[0];
#pragma unroll
    for (int q = 1; q < NW; ++q) b = umax64(b, s[q]);
    return b;
  } else {
    static_assert(NW <= 16, "one key per lane of a row");
    return wave_max_key<16>(lane < NW ? s[lane] : 0ull);
  }
}

// Orders lane 0's LDS writes before the wave's following LDS reads.
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---- small triangular solves on MFMA tiles ----------------------------------
constexpr int kTri = 64;

// One wave: the inverse of a 16 x 16 unit-lower block by forward
// substitution, the solved row broadcast by lane shuffles; lane l ends with
// rows 4q + l/16 of column l%16.  L(i, k) gives the entries below the diagonal.
template <typename F>
__device__ inline void tri_inv16(F&& L, double (*out)[17]) {
  const int lane = threadIdx.x & 63, c = lane & 15, r4 = lane >> 4;
  double y[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) y[q] = (4 * q + r4 == c) ? 1.0 : 0.0;
#pragma unroll
  for (int k = 0; k < 15; ++k) {
    const double xk = __shfl(y[k >> 2], ((k & 3) << 4) | c, 64);  // X[k][c]
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = 4 * q + r4;
      if (i > k) y[q] -= L(i, k) * xk;
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) out[4 * q + r4][c] = y[q];
}

// One wave: acc (four 16 x 16 tiles, rows 16 I of 16 columns, accumulator
// layout) <- inv(L) acc for the 64 x 64 unit-lower L, given its entries below
// the 16 x 16 diagonal blocks and those blocks' inverses.  An accumulator
// tile is the B operand of the next product as it stands: MFMA k-step s takes
// row row(lane, s), element s of the tile.  In FP64 for factors of either
// type, so that a solve or an inverse of FP32 factors is rounded once, at its
// end.
typedef Mma<double> MmaTri;
template <typename F>
__device__ inline void tri_solve64(MmaTri::acc_t (&acc)[4], F&& L, const double (*inv)[16][17]) {
  const int lane = threadIdx.x & 63, m = lane & 15;
#pragma unroll
  for (int I = 0; I < 4; ++I) {
#pragma unroll
    for (int J = 0; J < I; ++J)
#pragma unroll
      for (int s = 0; s < 4; ++s)
        acc[I] = MmaTri::mma(-(double)L(16 * I + m, 16 * J + MmaTri::row(lane, s)), acc[J][s], acc[I]);
    MmaTri::acc_t u = {};
#pragma unroll
    for (int s = 0; s < 4; ++s) u = MmaTri::mma(inv[I][m][MmaTri::row(lane, s)], acc[I][s], u);
    acc[I] = u;
  }
}

// Columns 64 q .. of row block v.b of the inverse (q <= v.b), by four waves:
// inv(L_bb) (-sum_{q <= k < b} L_bk X_kq), or inv(L_bb) itself for q = b.
// Operands come straight from memory: it runs beside the next leaf, or once
// at the panel's end.
template <typename T>
__device__ inline void inverse_rows(const InvArgs<T>& v, int q, double (*inv)[16][17]) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, m = lane & 15;
  const T* Lb = v.P + (int64_t)kTri * v.b * v.lda;  // rows of the block
  const T* D = Lb + kTri * v.b;
  // rows past the block read its last one and count as zero (in the diagonal
  // block columns past it read its first): loads inside the matrix without a
  // branch, which the compiler issues together
  auto entry = [&](const T* rows, int i, int k) -> T {
    const T x = rows[(int64_t)(i < v.w ? i : v.w - 1) * v.lda + k];
    return i < v.w ? x : T(0);
  };
  auto diag = [&](int i, int k) -> T { return entry(D, i, k < v.w ? k : 0); };
  tri_inv16([&](int i, int k) -> double { return (double)diag(16 * wv + i, 16 * wv + k); }, inv[wv]);
  __syncthreads();
  MmaTri::acc_t acc[4];
#pragma unroll
  for (int I = 0; I < 4; ++I)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      acc[I][e] = q == v.b && 16 * I + MmaTri::row(lane, e) == 16 * wv + m ? 1.0 : 0.0;
  const int c0 = kTri * q + 16 * wv + m;  // this lane's column of X
  for (int k = q; k < v.b; ++k) {
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      T bv[4], av[4][4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        // (any order of k serves both operands: FP32 entries in runs of four)
        const int kk = kTri * k + 16 * kb + Mma<T>::row(lane, s);
        bv[s] = v.X[(int64_t)kk * v.ldx + c0];
#pragma unroll
        for (int I = 0; I < 4; ++I) av[I][s] = entry(Lb, 16 * I + m, kk);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int I = 0; I < 4; ++I) acc[I] = MmaTri::mma(-(double)av[I][s], (double)bv[s], acc[I]);
    }
  }
  tri_solve64(acc, diag, inv);
#pragma unroll
  for (int I = 0; I < 4; ++I)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = 16 * I + MmaTri::row(lane, e);
      if (r < v.w && (q < v.b || 16 * wv + m < v.w)) v.X[(int64_t)(kTri * v.b + r) * v.ldx + c0] = (T)acc[I][e];
    }
}

// The W words of row q's candidate (tagged with tag) to lane c < n: entry c.
template <typename T>
__device__ inline void st_row_entry(unsigned long long* row, int c, T v, unsigned tag) {
  const unsigned long long t = (unsigned long long)tag << 32;
  if constexpr (sizeof(T) == 8) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    st_coh(row + 2 * c, (b & 0xFFFFFFFFull) | t);
    st_coh(row + 2 * c + 1, (b >> 32) | t);
  } else {
    st_coh(row + c, (unsigned long long)__float_as_uint(v) | t);
  }
}
template <typename T>
__device__ inline bool ld_row_entry(const unsigned long long* row, int c, unsigned tag, T& v) {
  if constexpr (sizeof(T) == 8) {
    const unsigned long long lo = ld_coh(row + 2 * c), hi = ld_coh(row + 2 * c + 1);
    v = __longlong_as_double((long long)((hi << 32) | (lo & 0xFFFFFFFFull)));
    return (unsigned)(lo >> 32) == tag && (unsigned)(hi >> 32) == tag;
  } else {
    const unsigned long long x = ld_coh(row + c);
    v = __uint_as_float((unsigned)x);
    return (unsigned)(x >> 32) == tag;
  }
}

// One leaf of the panel: columns [0, w) (w <= kPanelWMax) of rows [0, m) at
// a.A, factored by G workgroups of NT threads.  Thread t of workgroup g
// holds rows g*R + t + q*NT (q < ROWS) in registers.  The column loop runs
// over all kPanelWMax columns and rotates every row's registers left by one
// after each column, so the current column is always register 0 (no
// run-time register indexing) and after the loop the rows are back in
// column order.  Columns >= w are zero and only rotated.
//
// What bounds it is each column's chain of dependent steps, not its work:
// the workgroup's argmax, the staging of the best row, with G > 1 two trips
// of the exchange through the memory side of the chip (records, then the
// winner's row; a publish-to-poll trip is ~1.2 us), and the elimination.  So
// the row words carry their own tags (the row is not waited for before its
// record), the owner sends the reciprocal pivot along, one wave does the
// polling, the reduction takes 32-bit DPP steps, and the interchanges are
// replayed in registers.  One 64-wide leaf, averaged over the leaves of an
// LU, FP64 / FP32: 233 / 198 us at n = 10,000 (375 / 349 us with the row
// stored and waited for first, every thread polling, 64-bit DPP steps and
// the replay in LDS); FP32 at n = 40,000, beside the trailing update: 420 us
// (643 us).  The workgroups that form rows of the inverse cost registers:
// FP64 246 VGPRs with one row per thread (170 without), FP32 178 / 234 / 288
// with one / two / three rows (98 / 194 / 260), so an FP32 leaf of two or
// three rows per thread displaces one of the two update workgroups (2 x 152 of
// 512) on its CU.
template <typename T, int ROWS, int W, int NT>
__global__ __launch_bounds__(NT) void panel_kernel(PanelArgs<T> a) {
  static_assert(W <= kPanelWMax && W <= 64, "leaf wider than the candidate rows");
  // [0] this workgroup's candidate row of the current column, [1] the
  // winner's row: entry c belongs to column j + c, zeros from column w on.
  // The odd offset puts entry 1, the first one the elimination reads, on a
  // 16-byte boundary.
  constexpr int kOff = 16 / (int)sizeof(T) - 1;
  constexpr int NW = NT / 64;
  constexpr int kChunk = 8;
  constexpr int kRowLds = (kOff + W + 1 + 3) / 4 * 4;  // entry W: 1 / pivot
  __shared__ __align__(16) T s_row[2][kRowLds];
  __shared__ unsigned long long s_k1[NW], s_k2;
  __shared__ int s_win[W];
  __shared__ int s_zero[W];
  __shared__ int s_pos[W];

  const int G = a.G, g = blockIdx.x, tid = threadIdx.x;
  if constexpr (W > kPanelWNarrow) {
    // rows of the panel's inverse that the leaf before made possible
    if (g >= G) {
      __shared__ double s_inv[4][16][17];
      if (tid < 256) inverse_rows<T>(a.inv, g - G, s_inv);
      return;
    }
  }
  const int lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int w = a.w;
  const int64_t rb = (int64_t)g * a.R;
  const int64_t re = rb + a.R < a.m ? rb + a.R : a.m;
  const int nr = re > rb ? (int)(re - rb) : 0;

  T P[ROWS][W];
  // the column a row was chosen for, W while it is active, W + 1: no row
  int won[ROWS];
  // Rows are 512 bytes or less at a stride of lda, so a load of one entry
  // per lane touches 64 cache lines; 16-byte loads halve (FP64) or quarter
  // (FP32) the line visits.
  constexpr int E = 16 / (int)sizeof(T);
  typedef T vec_t __attribute__((ext_vector_type(E)));
  const bool wide = w == W && a.lda % E == 0 && (reinterpret_cast<uintptr_t>(a.A) & 15) == 0;
#pragma unroll
  for (int q = 0; q < ROWS; ++q) {
    const int local = tid + q * NT;
    won[q] = local < nr ? W : W + 1;
    const T* src = a.A + (rb + local) * a.lda;
    if (wide && local < nr) {
#pragma unroll
      for (int c = 0; c < W; c += E) {
        const vec_t x = *reinterpret_cast<const vec_t*>(src + c);
#pragma unroll
        for (int e = 0; e < E; ++e) P[q][c + e] = x[e];
      }
    } else {
#pragma unroll
      for (int c = 0; c < W; ++c) P[q][c] = (local < nr && c < w) ? src[c] : T(0);
    }
  }

  // key of this thread's best active row in register 0 (the current column)
  auto thread_key = [&]() -> unsigned long long {
    unsigned long long k = 0;
#pragma unroll
    for (int q = 0; q < ROWS; ++q)
      if (won[q] == W) k = umax64(k, pivot_key((double)fabs(P[q][0]), 0, tid + q * NT));
    return k;
  };
  unsigned long long* recs = reinterpret_cast<unsigned long long*>(a.cand);

  // rotate every row left by one: column j+1 into register 0, column j to
  // the top
  auto rotate = [&]() {
#pragma unroll
    for (int q = 0; q < ROWS; ++q) {
      const T t0 = P[q][0];
#pragma unroll
      for (int c = 0; c + 1 < W; ++c) P[q][c] = P[q][c + 1];
      P[q][W - 1] = t0;
    }
  };
  // bounded polling of one value by this lane; false when the factorisation
  // has failed elsewhere or the wait expired
  auto poll = [&](auto&& ready) -> bool {
    if (ready()) return true;
    uint32_t spins = 0;
    WaitClock clk(a.wait_ticks);
    for (;;) {
      __builtin_amdgcn_s_sleep(1);
      ++spins;
      if (ready()) return true;
      if ((spins & 255u) == 0 && __hip_atomic_load(a.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)
        return false;
      if (clk.expired()) {
        __hip_atomic_store(a.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return false;
      }
    }
  };
  // A leaf that stops early (a NaN column, an expired wait) moves no row: the
  // launches after it, already queued, index rows with its moves and pivots,
  // so workgroup 0 leaves well-formed ones on every way out.
  auto stop = [&]() {
    if (g != 0) return;
    if (tid < w) {
      a.ipiv[tid] = a.r0 + tid;
      a.moves[tid] = tid;
      a.moves[kPanelWMax + tid] = tid;
    }
    if (tid == 0) {
      a.moves[2 * kPanelWMax] = a.o;
      a.moves[2 * kPanelWMax + 1] = w;
    }
  };
  // the rows have arrived: without this the loop would wait for every memory
  // operation in flight at its top, the published row's stores included
  __builtin_amdgcn_s_waitcnt(0xF70);
  for (int j = 0; j < w; ++j) {
    // best active row of this workgroup for column j
    const unsigned long long k1 = block_max_key<NT>(thread_key(), s_k1);
    const int par = j & 1;
    const unsigned seq = a.seq_base + (unsigned)(j + 1);
    const unsigned long long tag = seq & 0xFFFFu;
    const int blocal = kKeyMaxRows - 1 - (int)(k1 & (kKeyMaxRows - 1));
    const int ow = k1 != 0 ? __builtin_amdgcn_readfirstlane((blocal % NT) >> 6) : 0;
    // 1. the wave that holds the best row stages it in LDS with its
    //    reciprocal pivot (the owning lane writes, then lane c reads entry c;
    //    a wave's LDS accesses stay in order) and, with other workgroups to
    //    tell, publishes it: the row in tagged words and, without waiting for
    //    those stores, the record
    //      w0 = bits of |value| with the 16 low mantissa bits set to the tag,
    //      w1 = tag << 48 | row.
    //    A reader takes a record only when both words carry the tag of
    //    column j, and a row entry only when its words do, so no store
    //    waits for another.  With no candidate, value -1 is published.
    if (k1 != 0 && wid == ow) {
      const int qo = blocal / NT;
      unsigned long long* row = a.cand_row + ((int64_t)par * G + g) * kRowStride<T>;
      if (G > 1 && lane == 0) {
        const double bv = __longlong_as_double((long long)(k1 & kKeyValMask));
        unsigned long long* rec = recs + kRecWords * ((int64_t)par * G + g);
        st_coh(rec, (unsigned long long)(__double_as_longlong(bv) & ~0xFFFFll) | tag);
        st_coh(rec + 1, (tag << 48) | ((unsigned long long)(rb + blocal) & 0xFFFFFFFFFFFFull));
      }
      T piv = T(0);
      if (lane == (blocal & 63)) {
#pragma unroll
        for (int q = 0; q < ROWS; ++q)
          if (q == qo) {
            piv = P[q][0];
#pragma unroll
            for (int c = 0; c < W; ++c) s_row[0][kOff + c] = P[q][c];
          }
      }
      wave_sync();
      if (lane < W && j + lane >= w) s_row[0][kOff + lane] = T(0);
      if (G > 1) {
        wave_sync();
        if (j + lane < w) st_row_entry(row, lane, s_row[0][kOff + lane], seq);
      }
      if (lane == (blocal & 63)) {
        const T rp = piv != T(0) ? T(1) / piv : T(0);
        if (G > 1)
          st_row_entry(row, kPanelWMax, rp, seq);
        else
          s_row[0][kOff + W] = rp;
      }
    } else if (G > 1 && k1 == 0 && tid == 0) {
      unsigned long long* rec = recs + kRecWords * ((int64_t)par * G + g);
      st_coh(rec, (unsigned long long)(__double_as_longlong(-1.0) & ~0xFFFFll) | tag);
      st_coh(rec + 1, (tag << 48) | 0xFFFFFFFFFFFFull);
    }
    // 2. one wave polls every workgroup's record of column j (a lane each),
    //    picks the winner (the same in every workgroup) and fetches its row;
    //    not the publishing wave, whose loads would wait for its stores
    if (G > 1 && wid == (ow + 1) % NW) {
      unsigned long long k2 = 0;
      bool ok = true;
      for (int q = lane; q < G; q += 64) {
        const unsigned long long* o = recs + kRecWords * ((int64_t)par * G + q);
        unsigned long long w0 = 0, w1 = 0;
        ok = ok && poll([&]() {
          w0 = ld_coh(o);
          w1 = ld_coh(o + 1);
          return (w0 & 0xFFFFull) == tag && (w1 >> 48) == tag;
        });
        const double ov = __longlong_as_double((long long)(w0 & ~0xFFFFull));
        if (ok && ov >= 0.0)
          k2 = umax64(k2, pivot_key(ov, q, (int)((int64_t)(w1 & 0xFFFFFFFFFFFFull) - (int64_t)q * a.R)));
      }
      k2 = wave_max_key(k2);
      const int wq = kKeyMaxGroups - 1 - (int)((k2 >> 11) & (kKeyMaxGroups - 1));
      if (k2 != 0 && wq < G) {
        T v = T(0), rp = T(0);
        if (j + lane < w) {
          const unsigned long long* row = a.cand_row + ((int64_t)par * G + wq) * kRowStride<T>;
          ok = ok && poll([&]() {
            const bool r1 = lane != 0 || ld_row_entry(row, kPanelWMax, seq, rp);
            return ld_row_entry(row, lane, seq, v) && r1;
          });
        }
        if (lane < W) s_row[1][kOff + lane] = v;
        if (lane == 0) s_row[1][kOff + W] = rp;
      }
      const bool bad = __ballot(!ok) != 0;
      if (lane == 0) s_k2 = bad ? kKeyBad : k2;
    }
    __syncthreads();
    const T* urow = &s_row[0][0] + (G > 1 ? kRowLds : 0) + kOff;
    const unsigned long long k2 = G > 1 ? s_k2 : k1;
    const T piv = urow[0], rpiv = urow[W];
    if (k2 == kKeyBad) {
      stop();
      return;
    }
    if (k2 == 0) {
      // no finite candidate anywhere (NaN column): every workgroup sees the
      // same key, so all of them leave here together
      if (g == 0 && tid == 0) {
        *a.info = -1;
        __hip_atomic_store(a.status, 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      stop();
      return;
    }
    const int wq = G > 1 ? kKeyMaxGroups - 1 - (int)((k2 >> 11) & (kKeyMaxGroups - 1)) : 0;
    const int wi = wq * (int)a.R + (kKeyMaxRows - 1 - (int)(k2 & (kKeyMaxRows - 1)));
    if (wq >= G || wi >= (int)a.m) {
      // a key that names no row cannot come from the records: stop
      if (tid == 0) __hip_atomic_store(a.status, 3, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      stop();
      return;
    }
    if (tid == 0) {
      s_win[j] = wi;
      s_zero[j] = piv == T(0);
    }
    // 3. eliminate column j from the active rows: register c holds column
    //    j + c (urow beyond w is zero, which also leaves the finished
    //    columns rotated to the top untouched).  Branch-free: an inactive
    //    row takes multiplier 0 (a divergent branch here makes the compiler
    //    keep a second copy of the row registers).  Eliminated and rotated
    //    in one pass: register c takes column j+1+c, the top register the
    //    multiplier of column j.
    T l[ROWS], top[ROWS];
#pragma unroll
    for (int q = 0; q < ROWS; ++q) {
      if ((int)rb + tid + q * NT == wi) won[q] = j;
      l[q] = won[q] == W ? P[q][0] * rpiv : T(0);
      top[q] = won[q] == W ? l[q] : P[q][0];
    }
#pragma unroll
    for (int c = 0; c + 1 < W; ++c) {
      // bounds the row entries held in registers ahead of their use
      if (c % kChunk == kChunk - 1) asm volatile("" ::: "memory");
      const T uc = urow[1 + c];
#pragma unroll
      for (int q = 0; q < ROWS; ++q) P[q][c] = P[q][c + 1] - l[q] * uc;
    }
#pragma unroll
    for (int q = 0; q < ROWS; ++q) P[q][W - 1] = top[q];
  }
  // the remaining rotations bring the columns back into register order
  for (int j = w; j < W; ++j) rotate();

  // Replay the interchanges (LAPACK order: at step j the rows at position j
  // and at the winner's position swap) to find every row's final position.
  // Only two kinds of row move: the leaf's first w rows, and winners from
  // below, each from its own place straight to its final position.  So lane
  // r of wave 0 keeps the position of row r and the row at position r.
  if (tid < 64) {
    const int win = lane < w ? s_win[lane] : 0;
    int pos = lane, occ = lane, from = 0;
    for (int j = 0; j < w; ++j) {
      const int p = __builtin_amdgcn_readlane(win, j);
      const int pp = p < w ? __builtin_amdgcn_readlane(pos, p) : p;  // position of the winner
      const int q = __builtin_amdgcn_readlane(occ, j);               // row at position j
      if (lane == q) pos = pp;
      if (lane == pp) occ = q;
      if (lane == p) pos = j;
      if (lane == j) from = pp;
    }
    if (lane < w) s_pos[lane] = pos;
    const unsigned long long z = __ballot(lane < w && s_zero[lane]);
    if (g == 0) {
      if (lane < w) {
        a.ipiv[lane] = a.r0 + from;
        a.moves[lane] = win;
        a.moves[kPanelWMax + lane] = pos;
      }
      if (lane == 0) {
        a.moves[2 * kPanelWMax] = a.o;
        a.moves[2 * kPanelWMax + 1] = w;
      }
      if (lane == 0 && z && *a.info == 0) *a.info = (int32_t)(a.r0 + __ffsll((long long)z));
    }
  }
  __syncthreads();
  // every row of this workgroup to its final position (the bound is hidden
  // from the compiler, which would keep the W column masks of the loads
  // alive in scalar registers until here)
  int wst = w;
  asm volatile("" : "+s"(wst));
#pragma unroll
  for (int q = 0; q < ROWS; ++q) {
    const int local = tid + q * NT;
    if (local >= nr) continue;
    const int64_t row = rb + local;
    const int64_t dest = won[q] < W ? won[q] : row < w ? s_pos[row] : row;
    T* dst = a.A + dest * a.lda;
    if (wide) {
#pragma unroll
      for (int c = 0; c < W; c += E) {
        vec_t x;
#pragma unroll
        for (int e = 0; e < E; ++e) x[e] = P[q][c + e];
        *reinterpret_cast<vec_t*>(dst + c) = x;
      }
    } else {
#pragma unroll
      for (int c = 0; c < W; ++c)
        if (c < wst) dst[c] = P[q][c];
    }
  }
}

// Inverse of the sz x sz (sz <= 64) unit-lower block at L into X[0:sz, 0:sz]
// (zeros above the diagonal included), in FP64 arithmetic.  Blocked by 16:
//   1. each wave inverts one 16 x 16 diagonal block by forward substitution,
//      the solved row broadcast across the wave by lane shuffles;
//   2. block rows I = 1..3 in turn: S = L[I, 0:I] X[0:I, 0:I], then
//      X[I, 0:I] = -X_II S (two barriers per block row).
// Rows and columns from sz to 64 are padded with the identity.
// NT = 16 for leaves of at most 16 columns: the 16 x 16 substitution alone.
template <typename T, int NT>
__device__ __forceinline__ void unit_inverse(const T* __restrict__ L, int64_t ldl, int sz,
                                                        T* __restrict__ X, int64_t ldx) {
  __shared__ double Ls[NT * (NT - 1) / 2];  // strictly lower part, packed by rows
  __shared__ double Xs[NT][NT + 1];
  __shared__ double Ss[16][NT + 1];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  auto lidx = [](int i, int k) { return i * (i - 1) / 2 + k; };
  // whole rows per pass (coalesced), all 16 loads in flight
  T lv[NT * NT / 256];
#pragma unroll
  for (int q = 0; q < NT * NT / 256; ++q) {
    const int e = q * 256 + t, i = e / NT, k = e % NT;
    lv[q] = (k < i && i < sz) ? L[(int64_t)i * ldl + k] : T(0);
  }
#pragma unroll
  for (int q = 0; q < NT * NT / 256; ++q) {
    const int e = q * 256 + t, i = e / NT, k = e % NT;
    if (k < i) Ls[lidx(i, k)] = (double)lv[q];
    Xs[i][k] = 0.0;
  }
  __syncthreads();
  if (16 * wv < NT) {
    const int c = lane & 15, r4 = lane >> 4, o = 16 * wv;
    double y[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) y[q] = (4 * q + r4 == c) ? 1.0 : 0.0;
#pragma unroll
    for (int k = 0; k < 15; ++k) {
      const double xk = __shfl(y[k >> 2], ((k & 3) << 4) | c, 64);  // X[k][c]
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int i = 4 * q + r4;
        if (i > k) y[q] -= Ls[lidx(o + i, o + k)] * xk;
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) Xs[o + 4 * q + r4][o + c] = y[q];
  }
  __syncthreads();
  for (int I = 1; I < NT / 16; ++I) {
    const int nI = 16 * I, oI = 16 * I;
    for (int e = t; e < 16 * nI; e += 256) {
      const int i = e / nI, j = e % nI;
      double acc = 0.0;
      for (int k = j; k < nI; ++k) acc += Ls[lidx(oI + i, k)] * Xs[k][j];  // X is lower: k >= j
      Ss[i][j] = acc;
    }
    __syncthreads();
    for (int e = t; e < 16 * nI; e += 256) {
      const int i = e / nI, j = e % nI;
      double acc = 0.0;
      for (int k = 0; k <= i; ++k) acc += Xs[oI + i][oI + k] * Ss[k][j];
      Xs[oI + i][j] = -acc;
    }
    __syncthreads();
  }
  for (int e = t; e < sz * sz; e += 256) {
    const int i = e / sz, c = e % sz;
    X[(int64_t)i * ldx + c] = (T)Xs[i][c];
  }
}

// A factored leaf's effect on the outer panel's other columns: its row
// interchanges, and on the columns to its right U12 = inv(L11) A12 of its
// rows.  A workgroup takes 64 columns: it reads the winners' rows (which
// become the leaf's rows) and the rows they displace, then writes both; on
// the right the winners' rows pass through the triangular solve first (16
// columns per wave, MFMA tiles, the 16 x 16 diagonal blocks inverted on the
// way).  Bound by the latency of its few dependent steps.  One launch instead of the
// interchanges inside the leaf, the inverse of its 64 x 64 block (20 us in one
// workgroup), a copy and one or two products per split of the panel.
// SOLVE false (recursive panels): the interchanges alone, and in the last
// workgroup the inverse of the leaf's diagonal block into ride.X.
template <typename T, bool SOLVE>
__global__ __launch_bounds__(256) void panel_apply_kernel(T* __restrict__ A, int64_t lda, int lcol, int w, int pw,
                                                          const int* __restrict__ moves, InvArgs<T> ride) {
  constexpr int LS = kTri + 16 / (int)sizeof(T);
  __shared__ T Ls[SOLVE ? kTri : 1][LS], Ss[SOLVE ? kTri : 1][kTri + 1];
  __shared__ double inv[4][16][17];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int nleft = (lcol + kTri - 1) / kTri;
  const int nright = (pw - lcol - w + kTri - 1) / kTri;
  if ((int)blockIdx.x >= nleft + nright) {
    if constexpr (SOLVE) {
      inverse_rows<T>(ride, (int)blockIdx.x - nleft - nright, inv);
    } else if (w <= 16) {
      unit_inverse<T, 16>(A + lcol, lda, w, ride.X, ride.ldx);
    } else {
      unit_inverse<T, kTri>(A + lcol, lda, w, ride.X, ride.ldx);
    }
    return;
  }
  const bool right = (int)blockIdx.x >= nleft;
  const int c0 = right ? lcol + w + ((int)blockIdx.x - nleft) * kTri : (int)blockIdx.x * kTri;
  const int nc = (right ? pw : lcol) - c0 < kTri ? (right ? pw : lcol) - c0 : kTri;
  T* C = A + c0;
  T vs[16], vd[16];
  int win[16], pos[16];
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const int r = wv + 4 * t;
    win[t] = r < w ? moves[r] : r;
    pos[t] = r < w ? moves[kPanelWMax + r] : r;
  }
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const int r = wv + 4 * t;
    vs[t] = r < w && lane < nc ? C[(int64_t)win[t] * lda + lane] : T(0);
    vd[t] = r < w && pos[t] >= w && lane < nc ? C[(int64_t)r * lda + lane] : T(0);
  }
  if (SOLVE && right) {
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      const int r = wv + 4 * t;
      Ls[r][lane] = r < w && lane < r ? A[(int64_t)r * lda + lcol + lane] : T(0);
    }
#pragma unroll
    for (int t = 0; t < 16; ++t) Ss[wv + 4 * t][lane] = vs[t];
  }
  // every row is in registers or LDS before any is overwritten
  __builtin_amdgcn_s_waitcnt(0xF70);
  __syncthreads();
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const int r = wv + 4 * t;
    if (r >= w || lane >= nc) continue;
    if (pos[t] >= w) C[(int64_t)pos[t] * lda + lane] = vd[t];
    if (!SOLVE || !right) C[(int64_t)r * lda + lane] = vs[t];
  }
  if (!SOLVE || !right) return;
  tri_inv16([&](int i, int k) -> double { return (double)Ls[16 * wv + i][16 * wv + k]; }, inv[wv]);
  __syncthreads();
  const int m = lane & 15;
  MmaTri::acc_t acc[4];
#pragma unroll
  for (int I = 0; I < 4; ++I)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[I][e] = Ss[16 * I + MmaTri::row(lane, e)][16 * wv + m];
  tri_solve64(
      acc, [&](int i, int k) -> T { return Ls[i][k]; }, inv);
  if (16 * wv + m >= nc) return;
#pragma unroll
  for (int I = 0; I < 4; ++I)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = 16 * I + MmaTri::row(lane, e);
      if (r < w) C[(int64_t)r * lda + 16 * wv + m] = (T)acc[I][e];
    }
}

// ---------------------------------------------------------------------------
// End of an outer panel of W columns at absolute row s, in one launch: the
// last row block of the inverse (workgroups 0 .. v.b), and the panel's net
// row interchange as (dst, src) pairs (the last workgroup), composed from
// the leaves' moves in order (moves[l]: winners and final positions of the
// first rows, relative to the leaf's first row, its column and width).  Each
// leaf's moves are one parallel step: content[t] is the row now at position
// t < W, and positions past the panel sit in a hash table once a winner came
// from there.  At most W positions are ever in the table, so a probe ends well
// before kPlanSlots steps; the loop is bounded all the same.  (Replaying the
// 512 interchanges one by one took 50-150 us.)
constexpr int kSwapMax = 512;
constexpr int kPlanSlots = 2048;

template <typename T>
__global__ __launch_bounds__(256) void panel_finish_kernel(InvArgs<T> v, const int* __restrict__ moves, int nl, int W,
                                                           int64_t s, int64_t* __restrict__ dst,
                                                           int64_t* __restrict__ src, int* __restrict__ count) {
  __shared__ double inv[4][16][17];
  __shared__ int content[kSwapMax];
  __shared__ int key[kPlanSlots], held[kPlanSlots];  // positions past the panel (-1: free), rows there
  __shared__ int nout;
  if ((int)blockIdx.x <= v.b) {
    inverse_rows<T>(v, blockIdx.x, inv);
    return;
  }
  const int tid = threadIdx.x;
  for (int t = tid; t < W; t += 256) content[t] = t;
  for (int t = tid; t < kPlanSlots; t += 256) key[t] = -1;
  if (tid == 0) nout = 0;
  __syncthreads();
  auto slot_of = [&](int p, bool insert) -> int {
    unsigned h = ((unsigned)p * 2654435761u) >> 21;
    for (int probe = 0; probe < kPlanSlots; ++probe, h = (h + 1) & (kPlanSlots - 1)) {
      const int k = key[h];
      if (k == p) return (int)h;
      if (insert && k == -1) {
        const int old = atomicCAS(&key[h], -1, p);
        if (old == -1) {
          held[h] = p;  // nothing moved there yet
          return (int)h;
        }
        if (old == p) return (int)h;
      }
    }
    return -1;
  };
  for (int l = 0; l < nl; ++l, moves += kMoveStride) {
    const int o = moves[2 * kPanelWMax], w = moves[2 * kPanelWMax + 1];
    int top = 0, low = 0, to = -1;
    if (tid < w) {
      const int p = o + moves[tid];
      const int at = p < W ? -1 : slot_of(p, true);
      top = p < W ? content[p] : at < 0 ? p : held[at];
      to = o + moves[kPanelWMax + tid];
      low = content[o + tid];
    }
    __syncthreads();
    if (tid < w) {
      content[o + tid] = top;
      // a displaced row goes where a winner from below the leaf came from
      if (to >= o + w) {
        const int at = to < W ? -1 : slot_of(to, false);
        if (to < W)
          content[to] = low;
        else if (at >= 0)
          held[at] = low;
      }
    }
    __syncthreads();
  }
  for (int t = tid; t < W; t += 256)
    if (content[t] != t) {
      const int k = atomicAdd(&nout, 1);
      dst[k] = s + t;
      src[k] = s + content[t];
    }
  for (int t = tid; t < kPlanSlots; t += 256)
    if (key[t] != -1 && held[t] != key[t]) {
      const int k = atomicAdd(&nout, 1);
      dst[k] = s + key[t];
      src[k] = s + held[t];
    }
  __syncthreads();
  if (tid == 0) *count = nout;
}

// This workgroup's share (blockIdx.x of gridDim.x) of a copy of nc
// entries, with 16-byte accesses when both ends are 16-byte aligned.
template <typename T>
__device__ inline void copy_row_part(const T* __restrict__ s, T* __restrict__ d, int64_t nc) {
  constexpr int E = 16 / sizeof(T);
  typedef T V __attribute__((ext_vector_type(E)));
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (((reinterpret_cast<uintptr_t>(s) | reinterpret_cast<uintptr_t>(d)) & 15) == 0) {
    const int64_t nv = nc / E;
    for (int64_t v = t0; v < nv; v += stride) reinterpret_cast<V*>(d)[v] = reinterpret_cast<const V*>(s)[v];
    for (int64_t c = nv * E + t0; c < nc; c += stride) d[c] = s[c];
  } else {
    for (int64_t c = t0; c < nc; c += stride) d[c] = s[c];
  }
}

template <typename T>
__global__ __launch_bounds__(256) void swap_gather_kernel(const T* __restrict__ A, int64_t lda,
                                                          int64_t c0, int64_t nc,
                                                          const int64_t* __restrict__ src,
                                                          const int* __restrict__ count,
                                                          T* __restrict__ tmp) {
  const int q = blockIdx.y;
  if (q >= *count) return;
  copy_row_part<T>(A + src[q] * lda + c0, tmp + (int64_t)q * nc, nc);
}

template <typename T>
__global__ __launch_bounds__(256) void swap_scatter_kernel(T* __restrict__ A, int64_t lda, int64_t c0,
                                                           int64_t nc,
                                                           const int64_t* __restrict__ dst,
                                                           const int* __restrict__ count,
                                                           const T* __restrict__ tmp) {
  const int q = blockIdx.y;
  if (q >= *count) return;
  copy_row_part<T>(tmp + (int64_t)q * nc, A + dst[q] * lda + c0, nc);
}

// ---------------------------------------------------------------------------
// U12 = inv(L11) A12 as one MFMA GEMM.  inv(L11) (unit lower, W <= kNB) is
// built with the panel, a row block per leaf.
constexpr int kNB = 512;  // outer panel width of the blocked LU

// dst (rows x cols, ld ldd) = src (ld lds)
template <typename T>
__global__ __launch_bounds__(256) void copy_block_kernel(const T* __restrict__ src, int64_t lds, int rows,
                                                        int64_t cols, T* __restrict__ dst, int64_t ldd) {
  const int r = blockIdx.y;
  for (int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x; c < cols; c += (int64_t)gridDim.x * 256)
    dst[(int64_t)r * ldd + c] = src[(int64_t)r * lds + c];
}

__global__ void zero_u32_kernel(unsigned* p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// A failed or timed-out panel launch leaves status != 0: report it as
// info = -1 (the factors are then invalid).
__global__ void status_to_info_kernel(const int* status, int32_t* info) {
  if (threadIdx.x == 0 && *status != 0) *info = -1;
}

// ---------------------------------------------------------------------------
// Driver.
// Scratch of one stream of the factorisation (row-swap plan and staging,
// inverse of the diagonal block).
template <typename T>
struct LuScratch {
  int64_t* plan_dst;
  int64_t* plan_src;
  int* plan_count;
  int64_t plan_s = -1, plan_e = -1;  // swap range whose plan is in plan_*
  T* swap_tmp;
  int64_t swap_tmp_elems;
  T* tri_inv;  // [kNB][kNB] inverse of the panel's diagonal block
};

template <typename T>
struct LuCtx {
  T* A;
  int64_t n, lda;
  int64_t* ipiv;
  int32_t* info;
  hipStream_t s;
  // workspace
  double* cand;     // [2][G_max] (|value|, row) records of the panel launches
  unsigned long long* cand_row;  // [2][kKeyMaxGroups][kRowStride<T>]
  int* status;
  unsigned seq;     // steps taken by the panel launches so far
  LuScratch<T> sc;
  int G_max;
  int wleaf = kPanelWMax;  // widest leaf
  bool recursive = false;  // panels by recursive halving (kRecursiveRows)
  T* panel_tmp = nullptr;  // [kNB][kNB] staging of the recursion
  int* moves = nullptr;  // [kMaxLeaves][kMoveStride] of the panel being factored
  int nleaves = 0;       // leaves factored so far in that panel (recursive panels)
};

// Upper bound on the workgroups of one leaf launch (0: the CU count).
static std::atomic<int> g_panel_groups{0};
constexpr int kPanelMaxRows = 3;  // rows per thread of the register-resident leaf

// A leaf short enough for one workgroup of up to 1024 (FP32) or 768 (FP64)
// rows, as many as its registers hold with one row per thread, is factored
// by that workgroup alone: no exchange.  All leaves of an n x n LU, one
// workgroup against 256-row workgroups: FP64 n = 512 1.75 / 1.90 ms, n = 768
// 2.52 / 2.62 ms; FP32 n = 450 1.29 / 1.39 ms, n = 1024 3.10 / 3.49 ms.
template <typename T>
static bool lone_leaf(int64_t m, int w, int& nt, LeafShape& shape) {
  constexpr int widest = sizeof(T) == 8 ? 768 : 1024;
  if (m > (w <= kPanelWNarrow ? kPanelThreads : widest)) return false;
  nt = m <= kPanelThreads ? kPanelThreads : m <= 512 ? 512 : widest;
  shape.rows = 1;
  shape.G = 1;
  shape.R = m;
  return true;
}

template <typename T>
static int leaf(LuCtx<T>& c, int64_t r0, int o, int w, int* moves, const InvArgs<T>& inv) {
  const DeviceInfo& di = device_info();
  const int64_t m = c.n - r0;
  int cap = g_panel_groups.load(std::memory_order_relaxed);
  if (cap <= 0 && sizeof(T) == 4) {
    // FP32: at most a quarter of the CUs (more only where three rows per
    // thread do not reach m).  Fewer workgroups, each with up to three rows
    // per thread, exchange faster beside the trailing update: 40k mixed step
    // 616 ms with up to 256 workgroups, 601 / 596 / 593 ms with 96 / 80 / 64.
    const int64_t need = ceil_div(m, (int64_t)kPanelThreads * kPanelMaxRows);
    cap = (int)std::max<int64_t>(di.num_cus / 4, need);
  }
  const int64_t gmax =
      std::min<int64_t>(cap > 0 ? std::min(cap, di.num_cus) : di.num_cus, kKeyMaxGroups - 1);
  // As few workgroups as one row per thread allows (every column's exchange
  // polls all G records); more rows per thread only when the CUs run out.
  LeafShape shape;
  // (a cap on the workgroups asks for the geometry below)
  int nt = kPanelThreads;
  if (!(g_panel_groups.load(std::memory_order_relaxed) == 0 && lone_leaf<T>(m, w, nt, shape))) {
    RBFX_REQUIRE(leaf_shape(m, gmax, nt, kPanelMaxRows, shape),
                 "matrix too large for the register-resident panel (m=%lld)", (long long)m);
  }
  const int rows = shape.rows;
  const int G = shape.G;
  const int64_t R = shape.R;
  PanelArgs<T> a;
  a.A = c.A + r0 * c.lda + r0;
  a.lda = c.lda;
  a.m = m;
  a.w = w;
  a.R = R;
  a.r0 = r0;
  a.G = G;
  a.moves = moves;
  a.o = o;
  a.inv = inv;
  RBFX_REQUIRE(w >= 1 && w <= kPanelWMax, "leaf width %d out of range", w);
  a.ipiv = c.ipiv + r0;
  a.cand = c.cand;
  a.cand_row = c.cand_row;
  a.seq_base = c.seq;
  a.status = c.status;
  a.info = c.info;
  a.wait_ticks = di.wait_ticks;
  RBFX_REQUIRE(G <= c.G_max && G < kKeyMaxGroups && R <= (int64_t)nt * rows && R < kKeyMaxRows,
               "too many panel workgroups or rows");
  const int pid = prof_start(sizeof(T) == 8 ? "panel_f64" : "panel_f32", c.s);
  // A plain launch on the panel stream.  The workgroups wait for each
  // other, which needs all G of them resident at once: G is at most the CU
  // count and a workgroup fits an empty CU, so the ones not yet resident
  // start as soon as the trailing-update workgroups on some CU retire;
  // every wait is bounded in any case.  (A cooperative launch guarantees
  // the same but goes through a separate device queue, which added ~60 us
  // of dispatch latency per leaf, measured.)
#define RBFX_LEAF(ROWS_, W_, NT_) \
  hipLaunchKernelGGL((panel_kernel<T, ROWS_, W_, NT_>), dim3(G + inv.b + 1), dim3(NT_), 0, c.s, a)
  if (nt != kPanelThreads) {
    if (nt == 512 && rows == 1) RBFX_LEAF(1, kPanelWMax, 512);
    else if (nt == 768 && rows == 1 && sizeof(T) == 8) RBFX_LEAF(1, kPanelWMax, sizeof(T) == 8 ? 768 : 512);
    else if (nt == 1024 && rows == 1 && sizeof(T) == 4) RBFX_LEAF(1, kPanelWMax, sizeof(T) == 4 ? 1024 : 512);
    else {
      set_error("no leaf kernel of %d threads and %d rows per thread", nt, rows);
      return RBFX_ERR_ARG;
    }
  } else if (w <= kPanelWNarrow) {
    if (rows == 1) RBFX_LEAF(1, kPanelWNarrow, kPanelThreads);
    else if (rows == 2) RBFX_LEAF(2, kPanelWNarrow, kPanelThreads);
    else RBFX_LEAF(3, kPanelWNarrow, kPanelThreads);
  } else {
    if (rows == 1) RBFX_LEAF(1, kPanelWMax, kPanelThreads);
    else if (rows == 2) RBFX_LEAF(2, kPanelWMax, kPanelThreads);
    else RBFX_LEAF(3, kPanelWMax, kPanelThreads);
  }
#undef RBFX_LEAF
  RBFX_CHECK_LAUNCH();
  prof_stop(pid, c.s, (double)m * w * w, 2.0 * sizeof(T) * m * w);
  c.seq += (unsigned)w;
  return RBFX_OK;
}

// Apply the swaps ipiv[s..e) to columns [c0, c0+nc).
template <typename T>
static int apply_swaps(LuCtx<T>& c, int64_t s, int64_t e, int64_t c0, int64_t nc) {
  if (nc <= 0 || e <= s) return RBFX_OK;
  RBFX_REQUIRE(c.sc.plan_s == s && c.sc.plan_e == e, "no plan of these interchanges");
  const int maxcnt = (int)(2 * (e - s));
  const int pid = prof_start("row_swaps", c.s);
  // process the columns in slices that fit the staging buffer
  const int64_t slice = std::max<int64_t>(256, c.sc.swap_tmp_elems / maxcnt);
  for (int64_t off = 0; off < nc; off += slice) {
    const int64_t w = std::min<int64_t>(slice, nc - off);
    // a workgroup moves at least 4 x 16 bytes per thread of a row
    dim3 grid((unsigned)std::min<int64_t>(ceil_div(w, 256 * 4 * (16 / (int64_t)sizeof(T))), 64), (unsigned)maxcnt);
    hipLaunchKernelGGL((swap_gather_kernel<T>), grid, dim3(256), 0, c.s, c.A, c.lda, c0 + off, w,
                       c.sc.plan_src, c.sc.plan_count, c.sc.swap_tmp);
    RBFX_CHECK_LAUNCH();
    hipLaunchKernelGGL((swap_scatter_kernel<T>), grid, dim3(256), 0, c.s, c.A, c.lda, c0 + off, w,
                       c.sc.plan_dst, c.sc.plan_count, c.sc.swap_tmp);
    RBFX_CHECK_LAUNCH();
  }
  prof_stop(pid, c.s, 0.0, 4.0 * sizeof(T) * (e - s) * nc);
  return RBFX_OK;
}

// Leading dimension of staged blocks: rows that the LDS-DMA product can read.
constexpr int64_t kStageAlign = 16;

// U12 = X A12 with X = inv(L11) of the W x W diagonal block at r0 (ld ldx)
// and columns [col, col+ncols): staged copy of A12, then one GEMM.
template <typename T>
static int trsm(LuCtx<T>& c, int64_t r0, int W, const T* X, int64_t ldx, int64_t col, int64_t ncols, T* tmp,
                int64_t tmp_elems) {
  if (ncols <= 0) return RBFX_OK;
  int st;
  const int pid = prof_start(sizeof(T) == 8 ? "trsm_f64" : "trsm_f32", c.s);
  T* B = c.A + r0 * c.lda + col;
  const int64_t slice = std::max<int64_t>((int64_t)GBN, tmp_elems / W / kStageAlign * kStageAlign);
  for (int64_t off = 0; off < ncols; off += slice) {
    const int64_t w = std::min<int64_t>(slice, ncols - off);
    const int64_t ldt = ceil_div(w, kStageAlign) * kStageAlign;
    hipLaunchKernelGGL((copy_block_kernel<T>), dim3((unsigned)std::min<int64_t>(ceil_div(w, 256), 64), W),
                       dim3(256), 0, c.s, B + off, c.lda, W, w, tmp, ldt);
    RBFX_CHECK_LAUNCH();
    if ((st = gemm_launch<T, 1>(W, w, W, T(1), X, ldx, tmp, ldt, T(0), B + off, c.lda, c.s, false, !c.recursive)))
      return st;
  }
  prof_stop(pid, c.s, 2.0 * W * W * ncols, 3.0 * sizeof(T) * W * ncols);
  return RBFX_OK;
}

// Factorisation of the panel rows [r0, n) x columns [r0, r0+W), leaf by leaf:
// each leaf's interchanges and triangular solve on the panel's other columns
// in one launch, then the rank-w update of the columns to its right.  It also
// leaves X = inv(L11) of the W x W unit-lower diagonal block (ld ldx) in X's
// lower triangle, 64 rows riding along with the leaf after them and the last
// ones with the interchange plan in out's plan buffers; X's strictly upper
// part must hold zeros (the buffer is cleared once per factorisation and
// only ever receives lower-triangular entries).
template <typename T>
static int panel(LuCtx<T>& c, int64_t r0, int W, T* X, int64_t ldx, LuScratch<T>& out) {
  int st;
  RBFX_REQUIRE(W <= kSwapMax && kTri % c.wleaf == 0, "panel too wide");
  InvArgs<T> inv;
  inv.P = c.A + r0 * c.lda + r0;
  inv.lda = c.lda;
  inv.X = X;
  inv.ldx = ldx;
  int nl = (W + c.wleaf - 1) / c.wleaf;
  if constexpr (sizeof(T) == 8) {
    if (c.recursive) {
      c.nleaves = 0;
      if ((st = panel_recursive(c, r0, W, r0, W, X, ldx))) return st;
      nl = c.nleaves;
    }
  }
  for (int o = 0, l = 0; !c.recursive && o < W; o += c.wleaf, ++l) {
    const int w = std::min(c.wleaf, W - o);
    const int rest = W - o - w;
    int* moves = c.moves + (size_t)l * kMoveStride;
    const bool whole = o > 0 && o % kTri == 0;  // the leaf before ended a row block
    inv.b = whole ? o / kTri - 1 : -1;
    inv.w = kTri;
    // (narrow leaves keep their registers low and leave the inverse to the
    // launch after them)
    InvArgs<T> ride = inv, none = inv;
    none.b = -1;
    if ((st = leaf(c, r0 + o, o, w, moves, w > kPanelWNarrow ? inv : none))) return st;
    if (w > kPanelWNarrow) ride.b = -1;
    if (o > 0 || rest > 0) {
      const int pid = prof_start(sizeof(T) == 8 ? "panel_apply_f64" : "panel_apply_f32", c.s);
      hipLaunchKernelGGL((panel_apply_kernel<T, true>), dim3((unsigned)(ceil_div(o, kTri) + ceil_div(rest, kTri) + ride.b + 1)),
                         dim3(256), 0, c.s, c.A + (r0 + o) * c.lda + r0, c.lda, o, w, W, (const int*)moves, ride);
      RBFX_CHECK_LAUNCH();
      prof_stop(pid, c.s, (double)w * w * rest, 4.0 * sizeof(T) * w * (W - w));
    }
    T* R = c.A + (r0 + o) * c.lda + r0 + o + w;  // the leaf's rows, columns to its right
    if ((st = gemm<T>(c.n - r0 - o - w, rest, w, T(-1), R + (int64_t)w * c.lda - w, c.lda, R, c.lda, T(1),
                      R + (int64_t)w * c.lda, c.lda, c.s, true)))
      return st;
  }
  inv.b = c.recursive ? -1 : (W - 1) / kTri;
  inv.w = W - kTri * inv.b;
  hipLaunchKernelGGL((panel_finish_kernel<T>), dim3(inv.b + 2), dim3(256), 0, c.s, inv, (const int*)c.moves, nl, W,
                     r0, out.plan_dst, out.plan_src, out.plan_count);
  RBFX_CHECK_LAUNCH();
  out.plan_s = r0;
  out.plan_e = r0 + W;
  return RBFX_OK;
}

// FP64 systems of at most this many rows take the recursive panels: U12 by
// the inverse of the half panel's whole diagonal block, as opposed to block
// substitution.  The limit keeps results, it buys neither speed nor accuracy:
// both forms are backward stable (same ||P A - L U||), and on 16 time
// steppings of 66 x 66 to 90 x 90 nodes neither is nearer to the 64-bit
// solution (median error of the gradients 2.0e-9 with either); but with kappa(K) ~
// 1e10 through tens of solves another rounding of the factors moves the
// results by up to 2e-9, and systems of this size keep theirs.  It costs 16.9
// against 15.4 ms at 4,096 and 4,097 unknowns; larger systems and the FP32
// factors (which only precondition) take the leaf-by-leaf panels: FP64 LU at
// n = 10,006 46.4 against 60.1 ms.
constexpr int64_t kRecursiveRows = 4096;
constexpr int kMaxLeaves = kNB / 8;  // the recursion splits no narrower than 8

// Recursive factorisation of the panel columns [r0, r0+W) of the outer panel
// that starts at column pc0 and is pw wide, X = inv(L11) as below; each half's
// inverse is joined with X21 = -X22 (L21 X11).
template <typename T>
static int panel_recursive(LuCtx<T>& c, int64_t pc0, int pw, int64_t r0, int W, T* X, int64_t ldx) {
  int st;
  if (W <= c.wleaf) {
    const int o = (int)(r0 - pc0);
    int* moves = c.moves + (size_t)c.nleaves++ * kMoveStride;
    RBFX_REQUIRE(c.nleaves <= kMaxLeaves, "too many leaves in a panel");
    InvArgs<T> v;
    if ((st = leaf(c, r0, o, W, moves, v))) return st;
    v.X = X;
    v.ldx = ldx;
    const int pid = prof_start("panel_apply_f64", c.s);
    hipLaunchKernelGGL((panel_apply_kernel<T, false>),
                       dim3((unsigned)(ceil_div(o, kTri) + ceil_div(pw - o - W, kTri) + 1)), dim3(256), 0, c.s,
                       c.A + r0 * c.lda + pc0, c.lda, o, W, pw, (const int*)moves, v);
    RBFX_CHECK_LAUNCH();
    prof_stop(pid, c.s, (double)W * W * W / 3.0, 4.0 * sizeof(T) * W * (pw - W));
    return RBFX_OK;
  }
  const int W1 = std::max(8, (W / 2 + 7) / 8 * 8);
  const int W2 = W - W1;
  if ((st = panel_recursive(c, pc0, pw, r0, W1, X, ldx))) return st;
  if ((st = trsm(c, r0, W1, X, ldx, r0 + W1, W2, c.panel_tmp, (int64_t)kNB * kNB))) return st;
  const int64_t m2 = c.n - r0 - W1;
  const T* L21 = c.A + (r0 + W1) * c.lda + r0;
  if ((st = gemm<T>(m2, W2, W1, T(-1), L21, c.lda, c.A + r0 * c.lda + r0 + W1, c.lda, T(1),
                    c.A + (r0 + W1) * c.lda + r0 + W1, c.lda, c.s, true, false)))
    return st;
  T* X22 = X + (int64_t)W1 * ldx + W1;
  if ((st = panel_recursive(c, pc0, pw, r0 + W1, W2, X22, ldx))) return st;
  // L21 (rows r0+W1 .. r0+W) is final now: later pivots only move rows
  // >= r0+W
  const int pid = prof_start("trtri_f64", c.s);
  if ((st = gemm_launch<T, 2>(W2, W1, W1, T(1), L21, c.lda, X, ldx, T(0), c.panel_tmp, W1, c.s, true, false)))
    return st;
  st = gemm_launch<T, 2>(W2, W1, W2, T(-1), X22, ldx, c.panel_tmp, W1, T(0), X + (int64_t)W1 * ldx, ldx, c.s, true,
                         false);
  prof_stop(pid, c.s, 2.0 * W2 * W1 * (double)(W1 + W2), (double)sizeof(T) * 3.0 * W1 * W2);
  return st;
}


static size_t getrf_ws_bytes(int64_t n, int bytes) {
  const int G = 1024;  // upper bound on workgroups of a leaf
  size_t b = 0;
  b += ws_round((size_t)2 * G * kRecWords * 8);   // cand records
  b += ws_round((size_t)2 * kKeyMaxGroups * (kPanelWMax + 2) * 2 * bytes);  // cand_row (tagged)
  b += ws_round(64);                              // status
  for (int q = 0; q < 2; ++q) {                   // two slots, filled by the panel stream in turn
    b += ws_round((size_t)2 * kSwapMax * 8) * 2;  // plan dst / src
    b += ws_round(64);                            // plan count
    b += ws_round((size_t)kNB * kNB * bytes);     // inverse of the diagonal block
  }
  // main stream: staging of row swaps (2*NB rows x min(n, 8192) columns) and
  // of the triangular solve's right-hand side (NB x n)
  b += ws_round((size_t)std::max<int64_t>(2 * kNB * std::min<int64_t>(n, 8192), (int64_t)kNB * ceil_div(n, kStageAlign) * kStageAlign) * bytes);
  b += ws_round((size_t)kMaxLeaves * kMoveStride * 4);  // moves of one panel's leaves
  b += ws_round((size_t)kNB * kNB * bytes);             // staging of the recursive panels
  return b;
}

template <typename T>
static bool carve_scratch(Workspace& ws, LuScratch<T>& sc, int64_t tmp_elems) {
  sc.plan_dst = ws.take<int64_t>(2 * kSwapMax);
  sc.plan_src = ws.take<int64_t>(2 * kSwapMax);
  sc.plan_count = ws.take<int>(16);
  sc.tri_inv = ws.take<T>((size_t)kNB * kNB);
  sc.swap_tmp_elems = tmp_elems;
  sc.swap_tmp = ws.take<T>(tmp_elems);
  sc.plan_s = sc.plan_e = -1;
  return sc.plan_dst && sc.plan_src && sc.plan_count && sc.tri_inv && (tmp_elems == 0 || sc.swap_tmp);
}

// The panels run on a second stream of this library (default priority, one
// per device) so that panel k+1 overlaps the trailing update of step k
// (look-ahead).  Enqueue sequences of concurrent calls on one device are
// serialised by a mutex, so the shared stream and events pair up correctly.
struct PanelStream {
  hipStream_t s = nullptr;
  hipEvent_t ev[2] = {nullptr, nullptr};
};
static std::mutex g_ps_mu;
static PanelStream g_ps[64];

// Releases the panel streams and events of every device (rbfx_shutdown).
int release_panel_streams() {
  std::lock_guard<std::mutex> lock(g_ps_mu);
  int dev0 = 0;
  RBFX_HIP(hipGetDevice(&dev0));
  for (int d = 0; d < 64; ++d) {
    PanelStream& p = g_ps[d];
    if (!p.s) continue;
    RBFX_HIP(hipSetDevice(d));
    RBFX_HIP(hipStreamSynchronize(p.s));
    for (int i = 0; i < 2; ++i) {
      if (p.ev[i]) RBFX_HIP(hipEventDestroy(p.ev[i]));
      p.ev[i] = nullptr;
    }
    RBFX_HIP(hipStreamDestroy(p.s));
    p.s = nullptr;
  }
  RBFX_HIP(hipSetDevice(dev0));
  return RBFX_OK;
}

static int panel_stream(PanelStream*& out) {
  int dev = 0;
  RBFX_HIP(hipGetDevice(&dev));
  RBFX_REQUIRE(dev >= 0 && dev < 64, "device index %d out of range", dev);
  PanelStream& p = g_ps[dev];
  if (!p.s) {
    RBFX_HIP(hipStreamCreateWithFlags(&p.s, hipStreamNonBlocking));
    for (int i = 0; i < 2; ++i) RBFX_HIP(hipEventCreateWithFlags(&p.ev[i], hipEventDisableTiming));
  }
  out = &p;
  return RBFX_OK;
}

template <typename T>
static int getrf(int64_t n, T* A, int64_t lda, int64_t* ipiv, void* work, size_t work_bytes,
                 int32_t* info, hipStream_t s) {
  RBFX_REQUIRE(n > 0 && lda >= n, "bad n / lda");
  RBFX_REQUIRE(A && ipiv && info, "null pointer");
  RBFX_REQUIRE(n < (int64_t)INT32_MAX, "n too large");
  RBFX_REQUIRE(work && work_bytes >= getrf_ws_bytes(n, sizeof(T)), "getrf workspace too small");
  const DeviceInfo& di = device_info();
  std::lock_guard<std::mutex> lock(g_ps_mu);
  PanelStream* ps = nullptr;
  int st;
  if ((st = panel_stream(ps))) return st;
  LuCtx<T> c;
  c.A = A;
  c.n = n;
  c.lda = lda;
  c.ipiv = ipiv;
  c.info = info;
  c.s = s;
  Workspace ws(work, work_bytes);
  const int G = 1024;
  c.cand = ws.take<double>((size_t)2 * G * kRecWords);
  constexpr size_t row_words = (size_t)2 * kKeyMaxGroups * kRowStride<T>;
  c.cand_row = ws.take<unsigned long long>(row_words);
  unsigned* ctl = ws.take<unsigned>(16);
  c.status = reinterpret_cast<int*>(ctl + 1);
  // main stream: two slots of (plan, inverse) filled by the panel stream
  // for alternate steps, one staging buffer
  LuScratch<T> slot[2];
  const int64_t tmp_main =
      std::max<int64_t>(2 * kNB * std::min<int64_t>(n, 8192), (int64_t)kNB * ceil_div(n, kStageAlign) * kStageAlign);
  bool ok = carve_scratch(ws, slot[0], tmp_main) && carve_scratch(ws, slot[1], 0);
  c.moves = ws.take<int>((size_t)kMaxLeaves * kMoveStride);
  c.panel_tmp = ws.take<T>((size_t)kNB * kNB);
  c.recursive = sizeof(T) == 8 && n <= kRecursiveRows;
  ok = ok && c.moves && c.panel_tmp;
  slot[1].swap_tmp = slot[0].swap_tmp;
  slot[1].swap_tmp_elems = slot[0].swap_tmp_elems;
  RBFX_REQUIRE(ok && c.cand && c.cand_row, "workspace carve failed");
  c.seq = 0;
  c.G_max = G;
  hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(64), 0, s, ctl, 16);
  RBFX_CHECK_LAUNCH();
  // pivot records and candidate rows start with tag 0, which no column uses
  hipLaunchKernelGGL(zero_u32_kernel, dim3(4 * G * kRecWords / 64), dim3(64), 0, s,
                     reinterpret_cast<unsigned*>(c.cand), 4 * G * kRecWords);
  RBFX_CHECK_LAUNCH();
  hipLaunchKernelGGL(zero_u32_kernel, dim3((unsigned)(2 * row_words / 256)), dim3(256), 0, s,
                     reinterpret_cast<unsigned*>(c.cand_row), (int)(2 * row_words));
  RBFX_CHECK_LAUNCH();
  hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(64), 0, s, reinterpret_cast<unsigned*>(info), 1);
  RBFX_CHECK_LAUNCH();
  // the diagonal-block inverses: strictly upper parts stay zero from here on
  for (int q = 0; q < 2; ++q) {
    const int words = (int)((size_t)kNB * kNB * sizeof(T) / 4);
    hipLaunchKernelGGL(zero_u32_kernel, dim3((unsigned)ceil_div(words, 256)), dim3(256), 0, s,
                       reinterpret_cast<unsigned*>(slot[q].tri_inv), words);
    RBFX_CHECK_LAUNCH();
  }

  // panel context: same matrix and pivot records, own stream and scratch
  LuCtx<T> cp = c;
  cp.s = ps->s;
  hipEvent_t ready = ps->ev[0], done = ps->ev[1];
  // Panel stream, per step: factor the panel (which also leaves the inverse
  // of its diagonal block in the main stream's slot), then the
  // row-interchange plan for that slot.
  // Narrow leaves only on request, and only for panels that run beside a
  // trailing update (not for panel 0, which runs alone).
  auto panel_step = [&](int64_t r0, int W, LuScratch<T>& out, bool beside_update) -> int {
    int e;
    const int pid = prof_start(sizeof(T) == 8 ? "panel_step_f64" : "panel_step_f32", cp.s);
    const int64_t nl = g_narrow_leaf_rows.load(std::memory_order_relaxed);
    cp.wleaf = beside_update && nl > 0 && n - r0 >= nl ? kPanelWNarrow : kPanelWMax;
    if ((e = panel(cp, r0, W, out.tri_inv, (int64_t)kNB, out))) return e;
    prof_stop(pid, cp.s, (double)(n - r0) * W * W, 0.0);
    return RBFX_OK;
  };
  // panel 0 after everything queued so far on the caller's stream
  RBFX_HIP(hipEventRecord(ready, s));
  RBFX_HIP(hipStreamWaitEvent(cp.s, ready, 0));
  if ((st = panel_step(0, (int)std::min<int64_t>(kNB, n), slot[0], false))) return st;
  RBFX_HIP(hipEventRecord(done, cp.s));
  int par = 0;
  for (int64_t k0 = 0; k0 < n; k0 += kNB, par ^= 1) {
    const int W = (int)std::min<int64_t>(kNB, n - k0);
    const int64_t k1 = k0 + W;
    const int64_t rest = n - k1;
    c.sc = slot[par];
    RBFX_HIP(hipStreamWaitEvent(s, done, 0));  // panel k0, its plan and inverse are ready
    if (rest <= 0) {
      if ((st = apply_swaps(c, k0, k1, 0, k0))) return st;
      break;
    }
    const T* L21 = A + k1 * lda + k0;
    const T* U12 = A + k0 * lda + k1;
    T* A22 = A + k1 * lda + k1;
    // The next panel's columns first (interchanges, U12 block, update): the
    // panel stream waits for exactly these.  It then factors that panel
    // while this stream does the rest of the step (look-ahead): the
    // interchanges of the columns left of the panel, which nothing in the
    // factorisation reads again, and those, U12 and the update of the
    // remaining columns.  The rest of the step is enqueued before the panel,
    // whose many small launches take the host a few ms: so the device never
    // waits for the host to reach the long update.
    const int Wn = (int)std::min<int64_t>(kNB, rest);
    if ((st = apply_swaps(c, k0, k1, k1, Wn))) return st;
    if ((st = trsm(c, k0, W, c.sc.tri_inv, (int64_t)kNB, k1, Wn, c.sc.swap_tmp, c.sc.swap_tmp_elems))) return st;
    if ((st = gemm<T>(rest, Wn, W, T(-1), L21, lda, U12, lda, T(1), A22, lda, s, false, !c.recursive))) return st;
    RBFX_HIP(hipEventRecord(ready, s));
    if ((st = apply_swaps(c, k0, k1, 0, k0))) return st;
    if (rest > Wn) {
      if ((st = apply_swaps(c, k0, k1, k1 + Wn, rest - Wn))) return st;
      if ((st = trsm(c, k0, W, c.sc.tri_inv, (int64_t)kNB, k1 + Wn, rest - Wn, c.sc.swap_tmp,
                     c.sc.swap_tmp_elems))) return st;
      if ((st = gemm<T>(rest, rest - Wn, W, T(-1), L21, lda, U12 + Wn, lda, T(1), A22 + Wn, lda, s, false,
                        !c.recursive)))
        return st;
    }
    RBFX_HIP(hipStreamWaitEvent(cp.s, ready, 0));
    if ((st = panel_step(k1, Wn, slot[par ^ 1], rest > Wn))) return st;
    RBFX_HIP(hipEventRecord(done, cp.s));
  }
  hipLaunchKernelGGL(status_to_info_kernel, dim3(1), dim3(64), 0, s, c.status, info);
  RBFX_CHECK_LAUNCH();
  return RBFX_OK;
}

// Exposed for the blocked triangular solves and tests.
int gemm_f64(int64_t m, int64_t n, int64_t k, double alpha, const double* A, int64_t lda,
             const double* B, int64_t ldb, double beta, double* C, int64_t ldc, hipStream_t s) {
  return gemm<double>(m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, s);
}
int gemm_f32(int64_t m, int64_t n, int64_t k, float alpha, const float* A, int64_t lda,
             const float* B, int64_t ldb, float beta, float* C, int64_t ldc, hipStream_t s) {
  return gemm<float>(m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, s);
}

}  // namespace rbfx

using namespace rbfx;

extern "C" int rbfx_set_panel_groups(int max_groups) {
  RBFX_REQUIRE(max_groups >= 0, "max_groups must be >= 0");
  g_panel_groups.store(max_groups, std::memory_order_relaxed);
  return RBFX_OK;
}

extern "C" int rbfx_set_narrow_leaf_rows(int64_t rows) {
  g_narrow_leaf_rows.store(rows, std::memory_order_relaxed);
  return RBFX_OK;
}

extern "C" size_t rbfx_getrf_workspace(int64_t n, int dtype_bytes) {
  if (n <= 0 || (dtype_bytes != 4 && dtype_bytes != 8)) return 0;
  return getrf_ws_bytes(n, dtype_bytes);
}

extern "C" int rbfx_getrf_f64(int64_t n, double* d_A, int64_t lda, int64_t* d_ipiv, void* d_work,
                              size_t work_bytes, int32_t* d_info, void* stream) {
  return getrf<double>(n, d_A, lda, d_ipiv, d_work, work_bytes, d_info, as_stream(stream));
}

extern "C" int rbfx_getrf_f32(int64_t n, float* d_A, int64_t lda, int64_t* d_ipiv, void* d_work,
                              size_t work_bytes, int32_t* d_info, void* stream) {
  return getrf<float>(n, d_A, lda, d_ipiv, d_work, work_bytes, d_info, as_stream(stream));
}

// Test hook: C = beta C + alpha A B with the MFMA kernel.
extern "C" int rbfx_gemm_f64(int64_t m, int64_t n, int64_t k, double alpha, const double* d_A,
                             int64_t lda, const double* d_B, int64_t ldb, double beta, double* d_C,
                             int64_t ldc, void* stream) {
  RBFX_REQUIRE(m >= 0 && n >= 0 && k >= 0 && d_A && d_B && d_C, "bad gemm args");
  RBFX_REQUIRE(beta == 0.0 || beta == 1.0, "beta must be 0 or 1");
  return gemm<double>(m, n, k, alpha, d_A, lda, d_B, ldb, beta, d_C, ldc, as_stream(stream));
}
extern "C" int rbfx_gemm_f32(int64_t m, int64_t n, int64_t k, float alpha, const float* d_A,
                             int64_t lda, const float* d_B, int64_t ldb, float beta, float* d_C,
                             int64_t ldc, void* stream) {
  RBFX_REQUIRE(m >= 0 && n >= 0 && k >= 0 && d_A && d_B && d_C, "bad gemm args");
  RBFX_REQUIRE(beta == 0.0f || beta == 1.0f, "beta must be 0 or 1");
  return gemm<float>(m, n, k, alpha, d_A, lda, d_B, ldb, beta, d_C, ldc, as_stream(stream));
}
