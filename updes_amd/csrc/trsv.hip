// K4: triangular solves with the LU factors (FP64 and FP32), A x = b and
// A^T x = b, for a single right-hand side.
//
// Replaces the solve phase of lineax QR (updes/operators.py:612-613) and the
// inv(A) @ v products (updes/assembly.py:410,430).  Blocked, synchronisation-
// free sweep: superblocks of 512 rows, 16 workgroups of 32 rows each, taken in
// dependency order from an atomic ticket; each workgroup folds in the
// off-diagonal tiles of the superblocks already solved, exchanges its
// accumulated values with the superblock's other workgroups, applies its rows
// of the precomputed inverse of the diagonal superblock and publishes its
// slice.  Row-major storage makes the no-transpose tiles row-contiguous and
// the transposed tiles column-coalesced.
#include <algorithm>
#include <climits>
#include <vector>

#include <mutex>

#include "common.h"
#include "sweep_order.h"

namespace rbfx {

int gemm_f64(int64_t m, int64_t n, int64_t k, double alpha, const double* A, int64_t lda, const double* B,
             int64_t ldb, double beta, double* C, int64_t ldc, hipStream_t s);

constexpr int TB = 64;  // block size of the sweep and of the diagonal inverses

__host__ __device__ inline int64_t imin64(int64_t a, int64_t b) { return a < b ? a : b; }

// ---- diagonal-block inverses ----------------------------------------------
// dinv[b][0] = inv(unit lower L_bb), dinv[b][1] = inv(U_bb), TB x TB row-major,
// identity-padded for the last partial block.  One wave per (block,
// triangle): lane c substitutes column c in registers (the loops unroll
// fully), the block's entries are LDS broadcasts.  Bound by the dependent
// chains of 2,016 FMAs and, for U, 64 divides.  At n = 603 this took 112 us
// when both triangles were substituted through LDS by one wave.
template <typename TF, int WHICH>
__device__ __forceinline__ void diag_inv_body(const TF* __restrict__ LU, int64_t lda, int64_t n, int64_t b,
                                              double (*S)[TB + 2], double* __restrict__ dinv) {
  typedef double T;
  const int64_t o = b * TB;
  const int sz = (int)imin64(TB, n - o);
  const int c = threadIdx.x;
#pragma unroll 16
  for (int i = 0; i < TB; ++i) S[i][c] = (i < sz && c < sz) ? (T)LU[(o + i) * lda + o + c] : (i == c ? T(1) : T(0));
  __syncthreads();
  T x[TB];
  if constexpr (WHICH == 0) {
    // L^-1 column c: x_i = -sum_{c<=k<i} L_ik x_k
#pragma unroll
    for (int i = 0; i < TB; ++i) {
      T s = 0;
#pragma unroll
      for (int k = 0; k < i; ++k)
        if (k >= c) s = __builtin_fma(S[i][k], x[k], s);
      x[i] = i == c ? T(1) : (i > c && i < sz) ? -s : T(0);
    }
  } else {
    // U^-1 column c: x_i = (delta_ic - sum_{k>i} U_ik x_k) / U_ii
#pragma unroll
    for (int i = TB - 1; i >= 0; --i) {
      T s = i == c ? T(1) : T(0);
#pragma unroll
      for (int k = i + 1; k < TB; ++k)
        if (k <= c) s = __builtin_fma(-S[i][k], x[k], s);
      x[i] = i > c ? T(0) : s / S[i][i];
    }
  }
  T* Xo = dinv + (b * 2 + WHICH) * TB * TB;
#pragma unroll
  for (int i = 0; i < TB; ++i) Xo[i * TB + c] = x[i];
}

template <typename TF>
__global__ __launch_bounds__(TB) void diag_inv_kernel(const TF* __restrict__ LU, int64_t lda, int64_t n,
                                                      double* __restrict__ dinv) {
  __shared__ __align__(16) double S[TB][TB + 2];
  const int64_t b = blockIdx.x >> 1;
  if (blockIdx.x & 1)
    diag_inv_body<TF, 1>(LU, lda, n, b, S, dinv);
  else
    diag_inv_body<TF, 0>(LU, lda, n, b, S, dinv);
}

// ---- permutation staging ------------------------------------------------------
// ctl[0] = ticket, ctl[1] = completion counter of the current sweep,
// ctl[2] = status of the whole solve (nonzero: a wait expired).  The solve's
// first gather clears all three; the reset before each sweep only the first
// two, so an expired wait in the first sweep survives the second.
__global__ void gather_perm_kernel(const double* __restrict__ b, const int64_t* __restrict__ perm,
                                   int64_t n, double* __restrict__ y, unsigned* __restrict__ ctl,
                                   int clear_status) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) {
    ctl[0] = 0u;
    ctl[1] = 0u;
    if (clear_status) ctl[2] = 0u;
  }
  if (i < n) y[i] = b[perm ? perm[i] : i];
}

// Writes the solution back; a solve whose status is set writes NaN instead,
// so that a timed-out solve never reads as a result.
__global__ void scatter_perm_kernel(const double* __restrict__ y, const int64_t* __restrict__ perm,
                                    int64_t n, double* __restrict__ b, const unsigned* __restrict__ ctl) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool failed = ctl[2] != 0u;
  if (i < n) b[perm ? perm[i] : i] = failed ? __builtin_nan("") : y[i];
}

// ---- superblock sweep ---------------------------------------------------------
// The chain of a blocked triangular solve is what bounds it at these sizes:
// every exchange between workgroups is a coherent store and a poll through the
// memory side of the chip (~1.2 us each).  The superblock
// sweep makes the chain n/SB steps instead of n/TB: the solution advances by
// SB = 512 rows at a time, each superblock's rows solved with its 512 x 512
// diagonal inverse (built once per factorisation by sbinv_kernel), by NCH
// workgroups of CH rows:
//   1. fold the tiles of the superblocks already solved, in solve order, into
//      private partial sums (the predecessor's solution from its published
//      values, earlier ones once the count of solved superblocks covers them);
//   2. publish the chunk's CH accumulated values b - sum;
//   3. once all NCH chunks of the superblock are in, apply rows of its
//      diagonal inverse to the superblock's SB values and publish the CH
//      solution entries.
// Every published value carries its own tag (two 64-bit words, each half of
// the value beside a tag that the reset before the sweep cleared), so an
// exchange is one trip, store to poll: the reader polls the values it needs,
// one per thread, with no counter, and the writer does not wait for its stores.
// The loads of the next product start between the values' departure and the
// wait for the others'.
// Tickets are taken in start order and each superblock has NCH consecutive
// tickets, so the peers a workgroup waits for in step 3 have all started
// before any workgroup of a later superblock: the waits always end.
constexpr int SB = 512;
constexpr int CH = 32;
constexpr int NCH = SB / CH;
constexpr int kCtlLine = 32;  // words per superblock control line

// 512 x 512 inverse of a diagonal superblock of L (unit lower, which = 0) or
// U (which = 1) in FP64, from the 64 x 64 inverses D_i of its sub-blocks:
//   lower:  X_ii = D_i,  X_ij = -D_i sum_{j<=k<i} L_ik X_kj   (i > j)
//   upper:  X_ii = D_i,  X_ij = -D_i sum_{i<k<=j} U_ik X_kj   (i < j)
// Columns of the inverse do not depend on each other, so a workgroup takes
// kInvCols columns of one 64-wide block column: the chain is at most 35
// products of a 64 x 64 tile with 64 x kInvCols values, kept in LDS, the next
// tile loading meanwhile.  Each thread sums a 2 x 2 patch in a fixed order.
// Rows and columns past n are identity.  With one workgroup per (superblock,
// triangle) doing all 112 products through memory this took 1.31 ms at
// n = 603 and 1.52 ms at n = 10,006.
constexpr int kInvCols = 16;
constexpr int kInvParts = TB / kInvCols;
template <typename TF>
__global__ __launch_bounds__(256) void sbinv_kernel(const TF* __restrict__ LU, int64_t lda, int64_t n,
                                                    const double* __restrict__ dinv64, double* __restrict__ dinv512) {
  constexpr int NSUB = SB / TB;
  constexpr int LX = kInvCols + 2;
  typedef double vd2 __attribute__((ext_vector_type(2)));
  __shared__ __align__(16) double Xs[SB][LX];  // the inverse's columns
  __shared__ __align__(16) double Ts[TB][LX];
  __shared__ __align__(16) double As[TB][TB + 2];
  const int part = blockIdx.x % kInvParts;
  const int j = (blockIdx.x / kInvParts) % NSUB;
  const int which = (blockIdx.x / (kInvParts * NSUB)) & 1;
  const int64_t K = blockIdx.x / (2 * kInvParts * NSUB);
  const int64_t o = K * SB;
  const int sz = (int)imin64(SB, n - o);
  const int nb = (sz + TB - 1) / TB;
  const double* D64 = dinv64 + ((o / TB) * 2 + which) * TB * TB;  // of sub-block b: D64 + 2 b TB^2
  const int tid = threadIdx.x;
  const int r0 = (tid >> 3) * 2, c0 = (tid & 7) * 2;
  const int lr = tid >> 6, lc = tid & 63;  // tile loads: rows lr + 4t, column lc
  // column block j: D_j, identity past the matrix
  for (int e = tid; e < SB * kInvCols; e += 256) {
    const int r = e / kInvCols, c = e % kInvCols;
    double v = 0.0;
    if (r / TB == j)
      v = j < nb ? D64[(int64_t)j * 2 * TB * TB + (r % TB) * TB + part * kInvCols + c]
                 : (r % TB == part * kInvCols + c ? 1.0 : 0.0);
    Xs[r][c] = v;
  }
  // The products in order: for each row block i away from the diagonal, the
  // tiles (i, k) of the factor with the blocks k between j and i, then D_i.
  // lower: rows below j; upper: rows above j, nearest first
  const int steps = j >= nb ? 0 : which == 0 ? nb - 1 - j : j;
  double ra[TB / 4];
  auto load_tile = [&](int step, int kk) {
    const int i = which == 0 ? j + step : j - step;
    if (kk < step) {
      // strictly lower / upper tile (i, k): no diagonal
      const int k = which == 0 ? j + kk : i + 1 + kk;
#pragma unroll
      for (int t = 0; t < TB / 4; ++t) {
        const int gr = i * TB + lr + 4 * t, gc = k * TB + lc;
        ra[t] = (gr < sz && gc < sz) ? (double)LU[(o + gr) * lda + o + gc] : 0.0;
      }
    } else {
#pragma unroll
      for (int t = 0; t < TB / 4; ++t) ra[t] = D64[(int64_t)i * 2 * TB * TB + (lr + 4 * t) * TB + lc];
    }
  };
  if (steps > 0) load_tile(1, 0);
  for (int step = 1; step <= steps; ++step) {
    const int i = which == 0 ? j + step : j - step;
    double acc[2][2] = {{0.0, 0.0}, {0.0, 0.0}};
    for (int kk = 0; kk <= step; ++kk) {
      __syncthreads();  // As free, Xs / Ts written
#pragma unroll
      for (int t = 0; t < TB / 4; ++t) As[lr + 4 * t][lc] = ra[t];
      __syncthreads();
      if (kk < step)
        load_tile(step, kk + 1);
      else if (step < steps)
        load_tile(step + 1, 0);
      const bool last = kk == step;  // X_ij = -D_i T
      const double* B = last ? &Ts[0][0] : &Xs[(which == 0 ? j + kk : i + 1 + kk) * TB][0];
      const double sign = last ? -1.0 : 1.0;
#pragma unroll 8
      for (int q = 0; q < TB; q += 2) {
        vd2 a[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) a[u] = *reinterpret_cast<const vd2*>(&As[r0 + u][q]);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const vd2 b = *reinterpret_cast<const vd2*>(B + (q + h) * LX + c0);
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            acc[u][0] = __builtin_fma(sign * a[u][h], b.x, acc[u][0]);
            acc[u][1] = __builtin_fma(sign * a[u][h], b.y, acc[u][1]);
          }
        }
      }
      if (kk >= step - 1) {
        double* dst = last ? &Xs[i * TB][0] : &Ts[0][0];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          *reinterpret_cast<vd2*>(dst + (r0 + u) * LX + c0) = vd2{acc[u][0], acc[u][1]};
          acc[u][0] = acc[u][1] = 0.0;
        }
      }
    }
  }
  __syncthreads();
  double* X = dinv512 + (K * 2 + which) * (int64_t)SB * SB + j * TB + part * kInvCols;
  for (int e = tid; e < SB * kInvCols; e += 256) X[(int64_t)(e / kInvCols) * SB + e % kInvCols] = Xs[e / kInvCols][e % kInvCols];
}

// Condition estimate of every diagonal superblock T_KK of L (which = 0, unit
// lower) and U (which = 1): max(||T||_inf ||X||_inf, ||T||_1 ||X||_1) with X
// its 512 x 512 inverse.  The FP64 sweeps apply X only where this is at most
// kCondRobust; above it they solve the block by substitution over its 64-row
// sub-blocks (one refinement step with X reduces the block residual by about
// kappa eps, so X serves a backward-stable solve only for kappa well below
// eps^-1/2).  kCondParts workgroups per (superblock, triangle) sum 64 rows
// and 64 columns each (coalesced: a wave per row, a lane per column), then
// one thread combines the parts.  0.49 ms at n = 603 when one workgroup
// summed a row and a column per thread.
constexpr double kCondRobust = 1e7;
constexpr int kCondParts = SB / 64;
constexpr int kCondThreads = 512;
template <typename TF>
__global__ __launch_bounds__(kCondThreads) void sbcond_part_kernel(const TF* __restrict__ LU, int64_t lda, int64_t n,
                                                                   const double* __restrict__ dinv512,
                                                                   double* __restrict__ part) {
  constexpr int NW = kCondThreads / 64;
  __shared__ double rows[2][NW], cols[2][NW][64];
  const int64_t blk = blockIdx.x / kCondParts;
  const int p0 = (int)(blockIdx.x % kCondParts) * 64;
  const int64_t I = blk >> 1;
  const int which = (int)(blk & 1);
  const int64_t o = I * SB;
  const int sz = (int)imin64(SB, n - o);
  const double* X = dinv512 + blk * (int64_t)SB * SB;
  const TF* F = LU + o * lda + o;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  auto entry = [&](int r, int c) -> double {  // |T[r][c]| (unit diagonal for L)
    if (which ? c < r : c > r) return 0.0;
    return which == 0 && c == r ? 1.0 : fabs((double)F[(int64_t)r * lda + c]);
  };
  double tr = 0, xr = 0;  // largest row sums of this wave
  for (int r = p0 + w; r < p0 + 64 && r < sz; r += NW) {
    double a = 0, x = 0;
#pragma unroll
    for (int t = 0; t < SB / 64; ++t) {
      const int c = lane + 64 * t;
      if (c < sz) {
        a += entry(r, c);
        x += fabs(X[(int64_t)r * SB + c]);
      }
    }
    for (int off = 32; off > 0; off >>= 1) {
      a += __shfl_xor(a, off, 64);
      x += __shfl_xor(x, off, 64);
    }
    tr = fmax(tr, a);
    xr = fmax(xr, x);
  }
  if (lane == 0) {
    rows[0][w] = tr;
    rows[1][w] = xr;
  }
  double tc = 0, xc = 0;  // this lane's column, the rows w, w + NW, ...
  const int c = p0 + lane;
  if (c < sz)
#pragma unroll 16
    for (int r = w; r < sz; r += NW) {
      tc += entry(r, c);
      xc += fabs(X[(int64_t)r * SB + c]);
    }
  cols[0][w][lane] = tc;
  cols[1][w][lane] = xc;
  __syncthreads();
  if (w < 2) {
    double v = 0, m = 0;
    for (int q = 0; q < NW; ++q) {
      v += cols[w][q][lane];
      m = fmax(m, rows[w][q]);
    }
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
    if (lane == 0) {
      part[blockIdx.x * 4 + 2 * w] = m;      // 0: T rows, 2: X rows
      part[blockIdx.x * 4 + 2 * w + 1] = v;  // 1: T columns, 3: X columns
    }
  }
}

__global__ void sbcond_kernel(int64_t nblk, const double* __restrict__ part, double* __restrict__ cond) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nblk) return;
  double m[4] = {0, 0, 0, 0};
  for (int p = 0; p < kCondParts; ++p)
    for (int e = 0; e < 4; ++e) m[e] = fmax(m[e], part[(b * kCondParts + p) * 4 + e]);
  cond[b] = fmax(m[0] * m[2], m[1] * m[3]);
}

// ctl[0] ticket, ctl[1] superblocks solved, ctl[2] status of the solve; the
// s-th processed superblock counts its solved chunks in word 3 of the
// 128-byte line ctl[kCtlLine (s + 1) ..].  Superblocks are counted in order
// (count_solved), so ctl[1] >= k means that the plain solution of superblocks
// 0 .. k-1 has arrived: what workgroups whose turn is far off poll (one thread
// each); the next superblock's workgroups poll their predecessor's solution
// itself.
// tags: four arrays of n published values (2n words each): solution,
// accumulated values, and for refined blocks first solution and residual.
//
// REFINE (FP64 factors): the inverse of an ill-conditioned 512 x 512
// diagonal block applied to the accumulated values loses digits that a
// substitution keeps (measured on the adjoint gradients, and as a backward
// error of 6e-9 against 8e-17 for substitution with the same factors of a
// numerically singular system).  In U blocks one step of refinement inside
// the block restores them for moderately conditioned blocks: x0 = D acc,
// r = acc - U_KK x0, x = x0 + D r, at two more exchanges per superblock.
// Blocks of L or U whose condition estimate exceeds kCondRobust are solved
// by substitution over their 64-row sub-blocks instead.  The FP32 factors of
// the preconditioner need neither: an application error there only perturbs
// the preconditioner.
constexpr int kSweepThreads = 512;
constexpr unsigned kTag = 1;         // tag of a published word (0: not yet)
constexpr int64_t kTagWords = 8;     // tagged words per row: four arrays of two words
constexpr int kSweepWaves = kSweepThreads / 64;
// Orders a wave's LDS writes before its following LDS reads.
__device__ inline void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename TF, bool FWD, bool TRANS, int WHICH, bool REFINE>
__global__ __launch_bounds__(kSweepThreads) void sbsweep_kernel(const TF* __restrict__ F, int64_t lda, int64_t n,
                                                                const double* __restrict__ D512,
                                                                const double* __restrict__ dinv64,
                                                                const double* __restrict__ cond, double* __restrict__ y,
                                                                unsigned long long* __restrict__ tags,
                                                                unsigned* __restrict__ ctl, uint64_t wait_ticks) {
  typedef double T;
  constexpr int RW = CH / kSweepWaves;        // chunk rows per wave (no-transpose)
  constexpr int NG = 2 * kSweepWaves;         // half-wave groups (transpose)
  constexpr int NV = SB * CH / kSweepThreads;  // operand values per thread
  constexpr int NP = TRANS ? 1 : RW;          // partial sums per thread
  static_assert(RW * kSweepWaves == CH && NV * NG == SB && NV == 8 * RW, "sweep layout");
  __shared__ T xs[SB];             // folded solution / accumulated values of the superblock
  __shared__ T xs2[SB];            // first solution, then its residual (REFINE)
  __shared__ T red[NG][CH + 1];    // cross-group partial sums
  __shared__ int s_t;
  __shared__ unsigned s_solved;
  __shared__ int s_failed;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int64_t nsb = ceil_div(n, SB);
  unsigned* ticket = ctl;
  unsigned* solved = ctl + 1;
  int* status = reinterpret_cast<int*>(ctl + 2);
  if (tid == 0) {
    s_t = (int)__hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_failed = 0;
    s_solved = 0;
    if (__hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) s_t = INT_MAX;
  }
  __syncthreads();
  const int t = s_t;
  if ((int64_t)t >= nsb * NCH) return;
  const int s = t / NCH, c = t % NCH;
  unsigned* parts = ctl + kCtlLine * (s + 1);
  const int64_t I = FWD ? s : nsb - 1 - s;
  const int64_t oI = I * SB;
  const int szI = (int)imin64(SB, n - oI);
  const int rc0 = c * CH;                                   // first row of the chunk in the superblock
  const int nr = szI - rc0 < 0 ? 0 : (szI - rc0 < CH ? szI - rc0 : CH);
  // Thread layout of every CH x SB operand, for the chunk's rows:
  //   no-transpose: wave w takes rows RW w .. RW w + RW-1, lane l the columns
  //     l, l+64, ..., l+448 (coalesced rows of the factor); reduced over the
  //     lanes;
  //   transpose: lane l & 31 takes chunk column l & 31, the NG half-waves
  //     g = 2w + (l >> 5) the rows NV g .. NV g + NV-1 of M[rows][chunk
  //     columns]; reduced over the half-waves.
  const int tcol = lane & 31, tgrp = 2 * w + (lane >> 5);

  // bounded polling of this thread; false if the solve failed.  far: not on
  // the critical path, poll less often
  auto wait_for = [&](auto&& ready, bool far) -> bool {
    if (ready()) return true;
    uint32_t spins = 0;
    WaitClock clk(wait_ticks);
    for (;;) {
      if (far)
        __builtin_amdgcn_s_sleep(8);
      else
        __builtin_amdgcn_s_sleep(1);
      ++spins;
      if (ready()) return true;
      if (clk.expired()) {
        __hip_atomic_store(status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return false;
      }
      if ((spins & 255u) == 0 && __hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)
        return false;
    }
  };
  // published values: entry i of array e
  auto publish = [&](int e, int64_t i, T v) {
    unsigned long long* w2 = tags + 2 * (e * n + i);
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    st_coh(w2, (b << 32) | kTag);
    st_coh(w2 + 1, (b & 0xFFFFFFFF00000000ull) | kTag);
  };
  auto published = [&](int e, int64_t i, T& v) -> bool {
    const unsigned long long* w2 = tags + 2 * (e * n + i);
    const unsigned long long lo = ld_coh(w2), hi = ld_coh(w2 + 1);
    v = __longlong_as_double((long long)((hi & 0xFFFFFFFF00000000ull) | (lo >> 32)));
    return (unsigned)lo == kTag && (unsigned)hi == kTag;
  };
  // stage the superblock's values of array e in dst (one per thread), waiting
  // for each; ends with a barrier
  static_assert(SB == kSweepThreads, "one published value per thread");
  auto collect = [&](int e, int64_t o, int sz, T* dst) -> bool {
    T v = T(0);
    if (tid < sz && !wait_for([&]() { return published(e, o + tid, v); }, false)) s_failed = 1;
    dst[tid] = v;
    __syncthreads();
    return s_failed == 0;
  };
  // reduce the per-thread partial sums of a product into red; after the
  // barrier, thread r < CH reads its row's value with row_value(r)
  auto reduce_rows = [&](T* ps) {
    if constexpr (!TRANS) {
#pragma unroll
      for (int k = 0; k < RW; ++k) {
        const T v = wave_sum(ps[k]);
        if (lane == 0) red[0][RW * w + k] = v;
      }
    } else {
      if (tid < NG * 32) red[tgrp][tcol] = ps[0];
    }
  };
  auto row_value = [&](int r) -> T {
    if constexpr (!TRANS) {
      return red[0][r];
    } else {
      T a = 0;
#pragma unroll
      for (int g = 0; g < NG; ++g) a += red[g][r];
      return a;
    }
  };
  // Loads of the operands are issued before the wait that releases their
  // use, so the chain of the sweep does not wait on HBM behind the other
  // workgroups' folds.
  // the factor's tile of column block oJ (szJ valid); diag: the stored
  // triangle of the diagonal block only (U_KK with its diagonal, or the
  // strictly lower part of the unit-lower L_KK; transposed as the sweep is)
  // Addresses are a wave-uniform base (scalar registers) plus one 32-bit
  // per-lane offset, so the NV loads in flight hold no vector address each.
  const int wu = __builtin_amdgcn_readfirstlane(w);
  const uint32_t hoff = (uint32_t)(lane >> 5) * NV;  // row offset of the upper half-wave (transpose)
  // Full tiles (every superblock but the last, off the diagonal) load
  // unmasked; the masks of the others compare against per-call limits, so no
  // per-value index is kept across the fold loop.
  auto load_F = [&](TF(&v)[NV], int64_t oJ, int szJ, bool diag) {
    const bool full = szJ == SB && nr == CH && !diag;
    if constexpr (!TRANS) {
      const int clim = szJ - lane;  // columns lane + 64m valid for 64m < clim
#pragma unroll
      for (int k = 0; k < RW; ++k) {
        const int r = RW * wu + k;
        const TF* row = F + (oI + rc0 + r) * lda + oJ;
        const int dlim = rc0 + r - lane;  // the diagonal entry: 64m == dlim
        if (full) {
#pragma unroll
          for (int m = 0; m < 8; ++m) v[8 * k + m] = row[(uint32_t)(lane + 64 * m)];
        } else if (r < nr) {
#pragma unroll
          for (int m = 0; m < 8; ++m) {
            const bool tri = WHICH == 1 ? 64 * m >= dlim : 64 * m < dlim;
            v[8 * k + m] = (64 * m < clim && (!diag || tri)) ? row[(uint32_t)(lane + 64 * m)] : TF(0);
          }
        } else {
#pragma unroll
          for (int m = 0; m < 8; ++m) v[8 * k + m] = TF(0);
        }
      }
    } else {
      const TF* base = F + (oJ + (int64_t)2 * wu * NV) * lda + oI + rc0;
      const uint32_t off = hoff * (uint32_t)lda + (uint32_t)tcol;
      if (full) {
#pragma unroll
        for (int q = 0; q < NV; ++q) v[q] = (base + q * lda)[off];
      } else {
        const int g0 = tgrp * NV;
        const int qlim = tcol < nr ? szJ - g0 : 0;  // rows g0 + q valid for q < qlim
        const int dlim = rc0 + tcol - g0;           // the diagonal entry: q == dlim
#pragma unroll
        for (int q = 0; q < NV; ++q) {
          const bool tri = WHICH == 1 ? q <= dlim : q > dlim;
          v[q] = (q < qlim && (!diag || tri)) ? (base + q * lda)[off] : TF(0);
        }
      }
    }
  };
  // rows of the superblock's diagonal inverse (columns for the transpose)
  const T* D = D512 + (I * 2 + WHICH) * (int64_t)SB * SB;
  auto load_D = [&](T(&v)[NV]) {
    if constexpr (!TRANS) {
#pragma unroll
      for (int k = 0; k < RW; ++k) {
        const int r = RW * wu + k;
        const T* row = D + (int64_t)(rc0 + r) * SB;
        if (r < nr) {
#pragma unroll
          for (int m = 0; m < 8; ++m) v[8 * k + m] = row[(uint32_t)(lane + 64 * m)];
        } else {
#pragma unroll
          for (int m = 0; m < 8; ++m) v[8 * k + m] = T(0);
        }
      }
    } else {
      const T* base = D + (int64_t)2 * wu * NV * SB + rc0;
      const uint32_t off = hoff * SB + (uint32_t)tcol;
      if (nr == CH) {
#pragma unroll
        for (int q = 0; q < NV; ++q) v[q] = (base + q * SB)[off];
      } else {
#pragma unroll
        for (int q = 0; q < NV; ++q) v[q] = tcol < nr ? (base + q * SB)[off] : T(0);
      }
    }
  };
  // ps += the operand held in v times the SB-vector vec (LDS), per thread
  auto product = [&](const auto& v, const T* vec, T* ps) {
    if constexpr (!TRANS) {
#pragma unroll
      for (int k = 0; k < RW; ++k) {
        T a = 0;
#pragma unroll
        for (int m = 0; m < 8; ++m) a = __builtin_fma((T)v[8 * k + m], vec[lane + 64 * m], a);
        ps[k] += a;
      }
    } else {
      T a = 0;
#pragma unroll
      for (int q = 0; q < NV; ++q) a = __builtin_fma((T)v[q], vec[tgrp * NV + q], a);
      ps[0] += a;
    }
  };
  auto apply = [&](const T(&dv)[NV], const T* vec) {
    T ps[NP];
#pragma unroll
    for (int k = 0; k < NP; ++k) ps[k] = 0;
    product(dv, vec, ps);
    reduce_rows(ps);
  };
  // publish the chunk's CH values into array e, start the loads that the next
  // product needs (they overlap the trip, and the values leave first), then
  // stage the superblock's SB values in dst
  auto exchange = [&](int e, T value, T* dst, auto&& loads) -> bool {
    if (tid < nr) publish(e, oI + rc0 + tid, value);
    loads();
    return collect(e, oI, szI, dst);
  };

  // 1. fold the superblocks solved before this one, in solve order.  The
  // predecessor's solution is polled value by value; earlier superblocks
  // through the solved count, so a workgroup that starts late folds them
  // without a poll each.  FP32 factors leave room to hold the diagonal
  // inverse's rows during the last wait as well; FP64 ones load them after
  // the fold.
  constexpr bool kEarlyD = sizeof(TF) == 4;
  T ps[NP];
#pragma unroll
  for (int k = 0; k < NP; ++k) ps[k] = 0;
  T dv[NV];
  if (kEarlyD && s == 0) load_D(dv);
  for (int d = 0; d < s; ++d) {
    const int64_t J = FWD ? d : nsb - 1 - d;
    const int64_t oJ = J * SB;
    const int szJ = (int)imin64(SB, n - oJ);
    TF tv[NV];
    load_F(tv, oJ, szJ, false);
    if (kEarlyD && d == s - 1) load_D(dv);
    __syncthreads();  // xs free
    if (d + 1 < s) {
      if (tid == 0 && s_solved <= (unsigned)d) {
        unsigned v = 0;
        if (!wait_for([&]() { return (v = ld_coh(solved)) >= (unsigned)(d + 1); }, true)) s_failed = 1;
        s_solved = v;
      }
      __syncthreads();
      if (s_failed) return;
      xs[tid] = tid < szJ ? ld_coh(y + oJ + tid) : T(0);  // complete: half the bytes of its tagged words
      __syncthreads();
    } else if (!collect(0, oJ, szJ, xs)) {
      return;
    }
    product(tv, xs, ps);
  }
  // 2. accumulated values b - (sum of the folded tiles); exchange them
  __syncthreads();
  reduce_rows(ps);
  __syncthreads();
  T acc_r = tid < nr ? y[oI + rc0 + tid] - row_value(tid) : T(0);
  if (!exchange(1, acc_r, xs, [&]() {
        if (!kEarlyD) load_D(dv);
      }))
    return;
  // 3. x = rows of D applied to the superblock's accumulated values
  T x;
  if constexpr (REFINE) {
    if (cond[I * 2 + WHICH] > kCondRobust) {
      // ill-conditioned block: every chunk solves the whole block by
      // substitution over its 64-row sub-blocks with their 64 x 64 inverses
      // (xs: values still to solve, xs2: solution), then keeps its rows.  The
      // next inverse, and the factor's entries four batches ahead, load while
      // the ones before are used.  A thread adds a row's terms in order; its
      // entries are coalesced in the transposed sweep, and in the other one
      // pass through the wave's part of ds (8 columns of 64 rows at a time).
      // 20-25 us a block; 60-95 us with every entry loaded when it was needed.
      __shared__ T ds[TB * (TB + 1)];
      constexpr int kBatch = TRANS ? 16 : 8, kAhead = TRANS ? 2 : 4;
      const int nsub = (szI + TB - 1) / TB;
      T dreg[TB * TB / kSweepThreads];
      auto load_inv = [&](int b) {
        const double* D64 = dinv64 + ((I * (SB / TB) + b) * 2 + WHICH) * (int64_t)(TB * TB);
#pragma unroll
        for (int q = 0; q < TB * TB / kSweepThreads; ++q) dreg[q] = D64[tid + q * kSweepThreads];
      };
      TF ent[kAhead][kBatch];
      // batch k of the columns of sub-block ob: this thread's row (TRANS), or
      // rows 8 q + lane / 8 of the wave's 64, column lane % 8
      auto load_batch = [&](int k, int ob, bool on) {
#pragma unroll
        for (int q = 0; q < kBatch; ++q) {
          TF& v = ent[k % kAhead][q];
          if constexpr (TRANS) {
            const int64_t j = oI + ob + k * kBatch + q;
            v = on && j < n && tid < szI ? F[j * lda + oI + tid] : TF(0);
          } else {
            const int64_t i = oI + 64 * w + 8 * q + (lane >> 3), j = oI + ob + k * kBatch + (lane & 7);
            v = on && i < n && j < n ? F[i * lda + j] : TF(0);
          }
        }
      };
      load_inv(FWD ? 0 : nsub - 1);
      for (int st = 0; st < nsub; ++st) {
        const int b = FWD ? st : nsub - 1 - st;
        const int ob = b * TB;
        const bool on = FWD ? w > b : w < b;  // (64 rows per wave: all of them or none)
#pragma unroll
        for (int q = 0; q < TB * TB / kSweepThreads; ++q) {
          const int e = tid + q * kSweepThreads;
          ds[e / TB * (TB + 1) + e % TB] = dreg[q];
        }
        if (st + 1 < nsub) load_inv(FWD ? b + 1 : b - 1);
#pragma unroll
        for (int k = 0; k < kAhead; ++k) load_batch(k, ob, on);
        __syncthreads();
        if (tid < TB) {
          T a = 0;
#pragma unroll 16
          for (int c2 = 0; c2 < TB; ++c2)
            a = __builtin_fma(ds[TRANS ? c2 * (TB + 1) + tid : tid * (TB + 1) + c2], xs[ob + c2], a);
          xs2[ob + tid] = ob + tid < szI ? a : T(0);
        }
        __syncthreads();
        if (on) {
          const int cend = szI - ob < TB ? szI - ob : TB;
          T* buf = ds + 64 * kBatch * w;
          T a = 0;
#pragma unroll
          for (int k = 0; k < TB / kBatch; ++k) {
            T v[kBatch];
            if constexpr (TRANS) {
#pragma unroll
              for (int q = 0; q < kBatch; ++q) v[q] = (T)ent[k % kAhead][q];
            } else {
              // (the xor spreads the 32 lanes of an access over the banks)
#pragma unroll
              for (int q = 0; q < kBatch; ++q) {
                const int r = 8 * q + (lane >> 3);
                buf[r * 8 + ((lane & 7) ^ ((r >> 2) & 7))] = (T)ent[k % kAhead][q];
              }
              wave_fence();
#pragma unroll
              for (int q = 0; q < kBatch; ++q) v[q] = buf[lane * 8 + (q ^ ((lane >> 2) & 7))];
              wave_fence();
            }
            if (k + kAhead < TB / kBatch) load_batch(k + kAhead, ob, on);
#pragma unroll
            for (int q = 0; q < kBatch; ++q)
              if (k * kBatch + q < cend) a = __builtin_fma(v[q], xs2[ob + k * kBatch + q], a);
          }
          if (tid < szI) xs[tid] -= a;
        }
        __syncthreads();
      }
      x = tid < nr ? xs2[rc0 + tid] : T(0);
      goto publish;
    }
  }
  apply(dv, xs);
  __syncthreads();
  x = tid < nr ? row_value(tid) : T(0);
  // the refinement step in U blocks; L blocks (unit diagonal, multipliers
  // at most 1) measured no better with it
  if constexpr (REFINE && WHICH == 1) {
    // x0 exchanged; r = acc - T_KK x0 (or T_KK^T x0) on the chunk's rows;
    // exchanged; x += D r.  The diagonal tile loads during the first
    // exchange, D's rows again during the second.
    TF uv[NV];
    if (!exchange(2, x, xs2, [&]() { load_F(uv, oI, szI, true); })) return;
    T pr[NP];
#pragma unroll
    for (int k = 0; k < NP; ++k) pr[k] = 0;
    product(uv, xs2, pr);
    __syncthreads();
    reduce_rows(pr);
    __syncthreads();
    const T r_r = tid < nr ? xs[rc0 + tid] - row_value(tid) : T(0);
    if (!exchange(3, r_r, xs2, [&]() { load_D(dv); })) return;
    apply(dv, xs2);
    __syncthreads();
    if (tid < nr) x += row_value(tid);
  }
publish:
  if (tid < nr) {
    publish(0, oI + rc0 + tid, x);
    st_coh(y + oI + rc0 + tid, x);
  }
  // (read while the stores drain: usually the predecessor is counted by now)
  const unsigned before = tid == 0 ? ld_coh(solved) : 0u;
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (tid == 0)
    count_solved(
        (unsigned)s, (unsigned)NCH,
        [&]() { return __hip_atomic_fetch_add(parts + 3, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); },
        [&](unsigned want) {
          return before >= want || wait_for([&]() { return ld_coh(solved) >= want; }, false);
        },
        [&](unsigned v) { st_coh(solved, v); });
}

// Clears the ticket, the superblocks' control lines and the tags of the four
// published arrays; the solve's status word ctl[2] stays.
__global__ __launch_bounds__(256) void reset_sweep_kernel(unsigned* ctl, int64_t nsb, unsigned long long* tags,
                                                          int64_t ntags) {
  typedef unsigned long long vu2 __attribute__((ext_vector_type(2)));
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < 2 || (i >= kCtlLine && i < kCtlLine * (nsb + 1))) ctl[i] = 0u;
  if (2 * i < ntags) reinterpret_cast<vu2*>(tags)[i] = vu2{0ull, 0ull};
}

// 64 x 64 inverses of L and U, then the 512 x 512 ones, then the condition
// estimates of the 512 x 512 blocks.
static int64_t dinv64_elems(int64_t n) { return ceil_div(n, TB) * 2 * TB * TB; }

template <typename T>
static int launch_sbsweep(bool fwd, bool trans, int which, const T* F, int64_t lda, int64_t n,
                          const double* dinv, double* y, unsigned long long* tags, unsigned* ctl, hipStream_t s) {
  const double* D512 = dinv + dinv64_elems(n);
  const double* cond = D512 + ceil_div(n, (int64_t)SB) * 2 * (int64_t)SB * SB;
  const int64_t nsb = ceil_div(n, (int64_t)SB);
  hipLaunchKernelGGL(reset_sweep_kernel,
                     dim3((unsigned)ceil_div(std::max<int64_t>(kCtlLine * (nsb + 1), kTagWords * n / 2), 256)), dim3(256),
                     0, s, ctl, nsb, tags, kTagWords * n);
  RBFX_CHECK_LAUNCH();
  const uint64_t ticks = device_info().wait_ticks;
  const unsigned grid = (unsigned)(nsb * NCH);
  const int pid = prof_start(sizeof(T) == 8 ? "sweep_f64" : "sweep_f32", s);
  // one refinement step in the diagonal blocks of FP64 factors
  constexpr bool R64 = sizeof(T) == 8;
#define RBFX_SBSWEEP(F_, T_, W_)                                                                              \
  hipLaunchKernelGGL((sbsweep_kernel<T, F_, T_, W_, R64>), dim3(grid), dim3(kSweepThreads), 0, s, F, \
                     lda, n, D512, dinv, cond, y, tags, ctl, ticks)
  if (fwd && !trans && which == 0) RBFX_SBSWEEP(true, false, 0);
  else if (!fwd && !trans && which == 1) RBFX_SBSWEEP(false, false, 1);
  else if (fwd && trans && which == 1) RBFX_SBSWEEP(true, true, 1);
  else if (!fwd && trans && which == 0) RBFX_SBSWEEP(false, true, 0);
  else {
    set_error("invalid sweep combination");
    return RBFX_ERR_ARG;
  }
#undef RBFX_SBSWEEP
  prof_stop(pid, s, (double)n * n, (double)sizeof(T) * n * (n + 1) / 2.0);
  RBFX_CHECK_LAUNCH();
  return RBFX_OK;
}

// Workspace of one solve: the permuted vector, the published values of a
// sweep, then the control words (3 + one line per superblock).
constexpr int64_t getrs_ctl_words(int64_t n) { return kCtlLine * ((n + SB - 1) / SB + 1) + 8; }
static bool carve_getrs(void* work, size_t work_bytes, int64_t n, double*& y, unsigned long long*& tags,
                        unsigned*& ctl) {
  Workspace ws(work, work_bytes);
  y = ws.take<double>(n);
  tags = ws.take<unsigned long long>(kTagWords * n);
  ctl = ws.take<unsigned>(getrs_ctl_words(n));
  return y && tags && ctl;
}

// The solve itself on carved scratch: y (n), tags (kTagWords n), ctl
// (getrs_ctl_words).
// Every scratch word that must start at zero is cleared by a kernel of the
// solve (no memset), and nothing is allocated.
template <typename T>
static int getrs_run(int trans, int64_t n, const T* LU, int64_t lda, const int64_t* perm, const double* dinv,
                     double* b, double* y, unsigned long long* tags, unsigned* ctl, hipStream_t s) {
  const unsigned g = (unsigned)ceil_div(n, 256);
  int st;
  if (!trans) {
    hipLaunchKernelGGL(gather_perm_kernel, dim3(g), dim3(256), 0, s, b, perm, n, y, ctl, 1);
    RBFX_CHECK_LAUNCH();
    if ((st = launch_sbsweep<T>(true, false, 0, LU, lda, n, dinv, y, tags, ctl, s))) return st;
    if ((st = launch_sbsweep<T>(false, false, 1, LU, lda, n, dinv, y, tags, ctl, s))) return st;
    hipLaunchKernelGGL(scatter_perm_kernel, dim3(g), dim3(256), 0, s, y, (const int64_t*)nullptr, n, b,
                       ctl);
    RBFX_CHECK_LAUNCH();
  } else {
    hipLaunchKernelGGL(gather_perm_kernel, dim3(g), dim3(256), 0, s, b, (const int64_t*)nullptr, n, y,
                       ctl, 1);
    RBFX_CHECK_LAUNCH();
    if ((st = launch_sbsweep<T>(true, true, 1, LU, lda, n, dinv, y, tags, ctl, s))) return st;
    if ((st = launch_sbsweep<T>(false, true, 0, LU, lda, n, dinv, y, tags, ctl, s))) return st;
    hipLaunchKernelGGL(scatter_perm_kernel, dim3(g), dim3(256), 0, s, y, perm, n, b, ctl);
    RBFX_CHECK_LAUNCH();
  }
  return RBFX_OK;
}

template <typename T>
static int getrs(int trans, int64_t n, const T* LU, int64_t lda, const int64_t* perm, const double* dinv,
                 double* b, void* work, size_t work_bytes, hipStream_t s) {
  RBFX_REQUIRE(n > 0 && lda >= n && LU && perm && dinv && b, "bad getrs args");
  RBFX_REQUIRE(n < (int64_t)INT32_MAX / 2, "getrs: n too large");
  double* y;
  unsigned long long* tags;
  unsigned* ctl;
  RBFX_REQUIRE(carve_getrs(work, work_bytes, n, y, tags, ctl), "getrs workspace too small");
  return getrs_run<T>(trans, n, LU, lda, perm, dinv, b, y, tags, ctl, s);
}


// ---- many right-hand sides -------------------------------------------------------
__global__ void gather_rows_kernel(const double* __restrict__ B, int64_t ldb, const int64_t* __restrict__ perm,
                                   int64_t n, int64_t nrhs, double* __restrict__ T, int64_t ldt) {
  const int64_t i = blockIdx.y;
  const int64_t src = perm[i];
  for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < nrhs; c += (int64_t)gridDim.x * blockDim.x)
    T[i * ldt + c] = B[src * ldb + c];
}

__global__ void copy_rows_kernel(const double* __restrict__ S, int64_t lds, int64_t rows, int64_t cols,
                                 double* __restrict__ D, int64_t ldd) {
  const int64_t i = blockIdx.y;
  if (i >= rows) return;
  for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < cols; c += (int64_t)gridDim.x * blockDim.x)
    D[i * ldd + c] = S[i * lds + c];
}

static size_t getrs_multi_ws(int64_t n, int64_t nrhs) {
  const int64_t ld = ceil_div(nrhs, 8) * 8;
  return ws_round(sizeof(double) * (size_t)n * ld) + ws_round(sizeof(double) * (size_t)TB * ld) + 256;
}

// A X = B for nrhs right-hand sides (B n x nrhs row-major, overwritten by X)
// with FP64 LU factors: rows gathered by the permutation, then blocked
// forward and backward substitution over the TB-row blocks, each block one
// MFMA GEMM against the blocks already solved and one with its precomputed
// diagonal inverse.
static int getrs_multi(int64_t n, const double* LU, int64_t lda, const int64_t* perm, const double* dinv,
                       int64_t nrhs, double* B, int64_t ldb, void* work, size_t work_bytes, hipStream_t s) {
  RBFX_REQUIRE(n > 0 && nrhs > 0 && lda >= n && ldb >= nrhs && LU && perm && dinv && B, "bad getrs_multi args");
  RBFX_REQUIRE(work && work_bytes >= getrs_multi_ws(n, nrhs), "getrs_multi workspace too small");
  const int64_t ldt = ceil_div(nrhs, 8) * 8;
  Workspace ws(work, work_bytes);
  double* T = ws.take<double>((size_t)n * ldt);
  double* W = ws.take<double>((size_t)TB * ldt);
  RBFX_REQUIRE(T && W, "getrs_multi workspace carve failed");
  const unsigned gx = (unsigned)std::min<int64_t>(ceil_div(nrhs, 256), 64);
  RBFX_REQUIRE(n < (int64_t)65536 * 65536, "getrs_multi: n too large");
  hipLaunchKernelGGL(gather_rows_kernel, dim3(gx, (unsigned)n), dim3(256), 0, s, B, ldb, perm, n, nrhs, T, ldt);
  RBFX_CHECK_LAUNCH();
  const int64_t nb = ceil_div(n, TB);
  int st;
  auto diag = [&](int64_t blk, int which) -> int {
    const int64_t o = blk * TB;
    const int64_t sz = imin64(TB, n - o);
    const double* D = dinv + (blk * 2 + which) * TB * TB;
    if ((st = gemm_f64(sz, nrhs, sz, 1.0, D, TB, T + o * ldt, ldt, 0.0, W, ldt, s))) return st;
    hipLaunchKernelGGL(copy_rows_kernel, dim3(gx, (unsigned)sz), dim3(256), 0, s, W, ldt, sz, nrhs, T + o * ldt, ldt);
    RBFX_CHECK_LAUNCH();
    return RBFX_OK;
  };
  for (int64_t blk = 0; blk < nb; ++blk) {  // L (unit lower)
    const int64_t o = blk * TB;
    const int64_t sz = imin64(TB, n - o);
    if (o > 0 && (st = gemm_f64(sz, nrhs, o, -1.0, LU + o * lda, lda, T, ldt, 1.0, T + o * ldt, ldt, s)))
      return st;
    if ((st = diag(blk, 0))) return st;
  }
  for (int64_t blk = nb - 1; blk >= 0; --blk) {  // U
    const int64_t o = blk * TB;
    const int64_t sz = imin64(TB, n - o);
    const int64_t e = o + sz;
    if (e < n && (st = gemm_f64(sz, nrhs, n - e, -1.0, LU + o * lda + e, lda, T + e * ldt, ldt, 1.0, T + o * ldt,
                                ldt, s)))
      return st;
    if ((st = diag(blk, 1))) return st;
  }
  hipLaunchKernelGGL(copy_rows_kernel, dim3(gx, (unsigned)n), dim3(256), 0, s, T, ldt, n, nrhs, B, ldb);
  RBFX_CHECK_LAUNCH();
  return RBFX_OK;
}

// Device word that a solve queued with this workspace sets when it fails.
const unsigned* getrs_failed(int64_t n, void* work, size_t work_bytes) {
  double* y;
  unsigned long long* tags;
  unsigned* ctl;
  return carve_getrs(work, work_bytes, n, y, tags, ctl) ? ctl + 2 : nullptr;
}

// Status of the last solve queued with this workspace (synchronises).
static int getrs_status(int64_t n, void* work, size_t work_bytes, hipStream_t s) {
  RBFX_REQUIRE(n > 0 && work, "bad getrs_status args");
  double* y;
  unsigned long long* tags;
  unsigned* ctl;
  RBFX_REQUIRE(carve_getrs(work, work_bytes, n, y, tags, ctl), "getrs workspace too small");
  unsigned st = 0;
  RBFX_HIP(hipMemcpyAsync(&st, ctl + 2, sizeof(st), hipMemcpyDeviceToHost, s));
  RBFX_HIP(hipStreamSynchronize(s));
  if (st != 0u) {
    set_error("triangular solve: a device-side wait expired after %.0f s (solution set to NaN)", kWaitSeconds);
    return RBFX_ERR_TIMEOUT;
  }
  return RBFX_OK;
}

template <typename T>
static int prepare(int64_t n, const T* LU, int64_t lda, const int64_t* ipiv, int64_t* perm, double* dinv,
                   hipStream_t s) {
  RBFX_REQUIRE(n > 0 && lda >= n && LU && ipiv && perm && dinv, "bad getrs_prepare args");
  std::vector<int64_t> hp(n), pm(n);
  RBFX_HIP(hipMemcpyAsync(hp.data(), ipiv, n * sizeof(int64_t), hipMemcpyDeviceToHost, s));
  RBFX_HIP(hipStreamSynchronize(s));
  // (checked before anything is queued)
  for (int64_t i = 0; i < n; ++i)
    RBFX_REQUIRE(hp[i] >= i && hp[i] < n, "invalid pivot ipiv[%lld] = %lld", (long long)i, (long long)hp[i]);
  // the inverses run while the host replays the interchanges
  const int64_t nsb = ceil_div(n, (int64_t)SB);
  double* d512 = dinv + dinv64_elems(n);
  double* cond = d512 + nsb * 2 * (int64_t)SB * SB;
  double* part = cond + 2 * nsb;
  hipLaunchKernelGGL((diag_inv_kernel<T>), dim3((unsigned)(2 * ceil_div(n, TB))), dim3(TB), 0, s, LU, lda, n, dinv);
  RBFX_CHECK_LAUNCH();
  hipLaunchKernelGGL((sbinv_kernel<T>), dim3((unsigned)(2 * nsb * (SB / TB) * kInvParts)), dim3(256), 0, s, LU, lda, n,
                     (const double*)dinv, d512);
  RBFX_CHECK_LAUNCH();
  hipLaunchKernelGGL((sbcond_part_kernel<T>), dim3((unsigned)(2 * nsb * kCondParts)), dim3(kCondThreads), 0, s, LU, lda,
                     n, (const double*)d512, part);
  RBFX_CHECK_LAUNCH();
  hipLaunchKernelGGL(sbcond_kernel, dim3((unsigned)ceil_div(2 * nsb, 256)), dim3(256), 0, s, 2 * nsb,
                     (const double*)part, cond);
  RBFX_CHECK_LAUNCH();
  for (int64_t i = 0; i < n; ++i) pm[i] = i;
  for (int64_t i = 0; i < n; ++i) std::swap(pm[i], pm[hp[i]]);
  RBFX_HIP(hipMemcpyAsync(perm, pm.data(), n * sizeof(int64_t), hipMemcpyHostToDevice, s));
  RBFX_HIP(hipStreamSynchronize(s));  // pm must outlive the copy
  return RBFX_OK;
}

}  // namespace rbfx

using namespace rbfx;

extern "C" size_t rbfx_getrs_multi_workspace(int64_t n, int64_t nrhs) {
  return (n <= 0 || nrhs <= 0) ? 0 : getrs_multi_ws(n, nrhs);
}

extern "C" int rbfx_getrs_multi_f64(int64_t n, const double* d_LU, int64_t lda, const int64_t* d_perm,
                                    const double* d_dinv, int64_t nrhs, double* d_B, int64_t ldb, void* d_work,
                                    size_t work_bytes, void* stream) {
  return getrs_multi(n, d_LU, lda, d_perm, d_dinv, nrhs, d_B, ldb, d_work, work_bytes, as_stream(stream));
}

extern "C" int64_t rbfx_getrs_dinv_elems(int64_t n) {
  return n <= 0 ? 0 : dinv64_elems(n) + ceil_div(n, (int64_t)SB) * (2 * (int64_t)SB * SB + 2 + 8 * kCondParts);
}

extern "C" size_t rbfx_getrs_workspace(int64_t n) {
  if (n <= 0) return 0;
  return ws_round((size_t)n * sizeof(double)) + ws_round((size_t)kTagWords * n * sizeof(unsigned long long)) +
         ws_round(getrs_ctl_words(n) * sizeof(unsigned)) + 512;
}

extern "C" int rbfx_getrs_prepare_f64(int64_t n, const double* d_LU, int64_t lda, const int64_t* d_ipiv,
                                      int64_t* d_perm, double* d_dinv, void* d_work, size_t work_bytes,
                                      void* stream) {
  (void)d_work;
  (void)work_bytes;
  return prepare<double>(n, d_LU, lda, d_ipiv, d_perm, d_dinv, as_stream(stream));
}

extern "C" int rbfx_getrs_prepare_f32(int64_t n, const float* d_LU, int64_t lda, const int64_t* d_ipiv,
                                      int64_t* d_perm, double* d_dinv, void* d_work, size_t work_bytes,
                                      void* stream) {
  (void)d_work;
  (void)work_bytes;
  return prepare<float>(n, d_LU, lda, d_ipiv, d_perm, d_dinv, as_stream(stream));
}

extern "C" int rbfx_getrs_f64(int trans, int64_t n, const double* d_LU, int64_t lda, const int64_t* d_perm,
                              const double* d_dinv, double* d_b, void* d_work, size_t work_bytes,
                              void* stream) {
  return getrs<double>(trans, n, d_LU, lda, d_perm, d_dinv, d_b, d_work, work_bytes, as_stream(stream));
}

namespace rbfx {
// ---- allocation-free solve ------------------------------------------------------
// Scratch of rbfx_getrs_noalloc_f64 for n <= RBFX_GETRS_NOALLOC_MAX_N, carved
// like a getrs workspace: y (n doubles), published values, control words.  One
// copy per device.  Host code never uses the symbol itself: its device
// address comes from hipGetSymbolAddress, once per device.
constexpr int64_t kNoAllocMaxN = RBFX_GETRS_NOALLOC_MAX_N;
constexpr size_t kNoAllocBytes = (1 + kTagWords) * (((size_t)kNoAllocMaxN * 8 + 255) / 256 * 256) +
                                 ((size_t)getrs_ctl_words(kNoAllocMaxN) * 4 + 255) / 256 * 256;
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];
static std::mutex g_scratch_mu;
static void* g_scratch_ptr[64];

static int scratch_address(void*& out) {
  int dev = 0;
  RBFX_HIP(hipGetDevice(&dev));
  RBFX_REQUIRE(dev >= 0 && dev < 64, "device index %d out of range", dev);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    RBFX_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    RBFX_REQUIRE(p != nullptr, "no device address for the solve's scratch array");
    g_scratch_ptr[dev] = p;
  }
  out = g_scratch_ptr[dev];
  return RBFX_OK;
}
}  // namespace rbfx

extern "C" int rbfx_getrs_noalloc_f64(int trans, int64_t n, const double* d_LU, int64_t lda,
                                      const int64_t* d_perm, const double* d_dinv, double* d_b, void* stream) {
  RBFX_REQUIRE(n > 0 && lda >= n && d_LU && d_perm && d_dinv && d_b, "bad getrs args");
  RBFX_REQUIRE(n <= kNoAllocMaxN, "rbfx_getrs_noalloc_f64: n = %lld exceeds its fixed scratch (n <= %lld)",
               (long long)n, (long long)kNoAllocMaxN);
  void* base = nullptr;
  int st;
  if ((st = scratch_address(base))) return st;
  double* y;
  unsigned long long* tags;
  unsigned* ctl;
  RBFX_REQUIRE(carve_getrs(base, kNoAllocBytes, n, y, tags, ctl), "solve scratch too small");
  return getrs_run<double>(trans, n, d_LU, lda, d_perm, d_dinv, d_b, y, tags, ctl, as_stream(stream));
}

extern "C" int rbfx_getrs_status(int64_t n, void* d_work, size_t work_bytes, void* stream) {
  return getrs_status(n, d_work, work_bytes, as_stream(stream));
}

extern "C" int rbfx_getrs_f32(int trans, int64_t n, const float* d_LU, int64_t lda, const int64_t* d_perm,
                              const double* d_dinv, double* d_b, void* d_work, size_t work_bytes,
                              void* stream) {
  return getrs<float>(trans, n, d_LU, lda, d_perm, d_dinv, d_b, d_work, work_bytes, as_stream(stream));
}
