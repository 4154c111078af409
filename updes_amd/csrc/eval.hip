// K6: evaluation of a field given by its RBF + monomial coefficients, and its
// transpose.  Reference: updes/operators.py:118-150 (value), 156-187
// (gradient), 319-351 (laplacian): a sum over ALL N centres (the evaluation
// point itself included, phi(0) for the value and 0 for derivatives) plus the
// monomial tail.  One block owns a few points, its threads stride over the
// centres, and a block reduction sums.
#include "common.h"
#include "rbf_device.h"

namespace rbfx {

constexpr int kEvThreads = 256;
constexpr int kEvPts = 4;

// What one (point, centre) pair contributes.  One operator at a time is the
// usual call (value, one component of the gradient, the Laplacian): the
// kernel then forms that operator alone, with r from the square-root
// sequence without range scaling where every r^2 of the wave allows it (the
// same bits as sqrt; NaN and extreme distances take sqrt itself).  kSetBoth is
// both components of the gradient from one square root, kSetAll all seven.
enum OpSet { kSetVal = 0, kSetGrad = 1, kSetLap = 2, kSetAll = 3, kSetBoth = 4 };

__host__ inline int op_set(uint32_t mask) {
  switch (mask) {
    case 1u << RBFX_VAL: return kSetVal;
    case 1u << RBFX_DX:
    case 1u << RBFX_DY: return kSetGrad;
    case 1u << RBFX_LAP: return kSetLap;
    case (1u << RBFX_DX) | (1u << RBFX_DY): return kSetBoth;
    default: return kSetAll;
  }
}

__device__ inline bool mid_or_zero(double r2) { return r2 == 0.0 || (r2 >= 0x1p-900 && r2 <= 0x1p900); }

// The operator of SET (kSetGrad: the component along d, which is dx or dy) at
// distance r, as all_ops forms it.
template <int SET>
__device__ inline double pair_op(const Kern& k, double r, double d) {
  if constexpr (SET == kSetVal) return radial_value(k, r);
  double phi, f1, g2;
  if (r == 0.0) return 0.0;
  radial(k, r, phi, f1, g2);
  return SET == kSetGrad ? f1 * d : g2 + 2.0 * f1;
}

// Sums of SET over `count` partners of PTS points, this thread's share: acc[q]
// += w_j op(d_qj), d = own - partner, or partner - own (FLIP).
template <int SET, int PTS, bool FLIP>
__device__ inline void pair_sums(const Kern& k, int64_t count, const double* __restrict__ ox,
                                 const double* __restrict__ oy, const double* __restrict__ w, const double (&px)[PTS],
                                 const double (&py)[PTS], bool along_y, double (&acc)[PTS]) {
  for (int64_t j = threadIdx.x; j < count; j += kEvThreads) {
    const double wj = w[j], xj = ox[j], yj = oy[j];
    double dx[PTS], dy[PTS], r2[PTS];
    bool mid = true;
#pragma unroll
    for (int q = 0; q < PTS; ++q) {
      dx[q] = FLIP ? xj - px[q] : px[q] - xj;
      dy[q] = FLIP ? yj - py[q] : py[q] - yj;
      r2[q] = dist2(dx[q], dy[q]);
      mid = mid && mid_or_zero(r2[q]);
    }
    if (__all(mid)) {
#pragma unroll
      for (int q = 0; q < PTS; ++q) {
        const double r = r2[q] > 0.0 ? sqrt_mid(r2[q]) : 0.0;
        acc[q] += wj * pair_op<SET>(k, r, along_y ? dy[q] : dx[q]);
      }
    } else {
#pragma unroll
      for (int q = 0; q < PTS; ++q) acc[q] += wj * pair_op<SET>(k, sqrt(r2[q]), along_y ? dy[q] : dx[q]);
    }
  }
}

template <int PTS, int LD>
__device__ inline void block_sums(const double (&acc)[PTS], double (*red)[LD]) {
  static_assert(LD >= kEvThreads / 64, "a sum per wave");
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q < PTS; ++q) {
    double v = acc[q];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    if (lane == 0) red[q][wid] = v;
  }
  __syncthreads();
}

// One operator (op, in SET) at PTS points per workgroup.  Bound by the FP64
// work of a pair (square root and about ten operations): 0.45 ms for one
// component at 40,007 points of a field of 10,000 centres, 1.38 ms when every
// call formed all seven operators (r^3).
template <int KIND, bool FAST, int SET, int PTS>
__global__ __launch_bounds__(kEvThreads) void eval_op_kernel(Kern k, int64_t N, int64_t M,
                                                             const double* __restrict__ cx,
                                                             const double* __restrict__ cy,
                                                             const double* __restrict__ coeffs, int64_t npts,
                                                             const double* __restrict__ px,
                                                             const double* __restrict__ py, int op,
                                                             double* __restrict__ out) {
  pin_kind<KIND, FAST>(k);
  const int64_t p0 = (int64_t)blockIdx.x * PTS;
  double xp[PTS], yp[PTS], acc[PTS];
#pragma unroll
  for (int q = 0; q < PTS; ++q) {
    const int64_t p = p0 + q < npts ? p0 + q : npts - 1;
    xp[q] = px[p];
    yp[q] = py[p];
    acc[q] = 0.0;
  }
  pair_sums<SET, PTS, false>(k, N, cx, cy, coeffs, xp, yp, op == RBFX_DY, acc);
  __shared__ double red[PTS][kEvThreads / 64];
  block_sums(acc, red);
  if (threadIdx.x < PTS) {
    const int q = threadIdx.x;
    if (p0 + q >= npts) return;
    double x = xp[0], y = yp[0];
#pragma unroll
    for (int e = 1; e < PTS; ++e)
      if (q == e) {
        x = xp[e];
        y = yp[e];
      }
    double s = 0.0;
    for (int w = 0; w < kEvThreads / 64; ++w) s += red[q][w];
    for (int64_t m = 0; m < M; ++m) {
      double o[RBFX_NOPS];
      mono_ops((int)m, x, y, o);
      s += coeffs[N + m] * o[op];
    }
    out[(int64_t)op * npts + p0 + q] = s;
  }
}

// Both components of the gradient (the same sums) from one square root: 0.43 ms
// at 40,007 points and 10,000 centres (r^3), two kernels of one component 0.92 ms;
// at 33 points of 600 centres one launch of 13 us instead of two.
template <int KIND, bool FAST, int PTS>
__global__ __launch_bounds__(kEvThreads) void eval_grad_kernel(Kern k, int64_t N, int64_t M,
                                                               const double* __restrict__ cx,
                                                               const double* __restrict__ cy,
                                                               const double* __restrict__ coeffs, int64_t npts,
                                                               const double* __restrict__ px,
                                                               const double* __restrict__ py,
                                                               double* __restrict__ out) {
  pin_kind<KIND, FAST>(k);
  const int64_t p0 = (int64_t)blockIdx.x * PTS;
  double xp[PTS], yp[PTS], acc[2 * PTS];
#pragma unroll
  for (int q = 0; q < PTS; ++q) {
    const int64_t p = p0 + q < npts ? p0 + q : npts - 1;
    xp[q] = px[p];
    yp[q] = py[p];
    acc[q] = acc[PTS + q] = 0.0;
  }
  for (int64_t j = threadIdx.x; j < N; j += kEvThreads) {
    const double wj = coeffs[j], xj = cx[j], yj = cy[j];
    double dx[PTS], dy[PTS], r[PTS];
    bool mid = true;
#pragma unroll
    for (int q = 0; q < PTS; ++q) {
      dx[q] = xp[q] - xj;
      dy[q] = yp[q] - yj;
      r[q] = dist2(dx[q], dy[q]);
      mid = mid && mid_or_zero(r[q]);
    }
    if (__all(mid)) {
#pragma unroll
      for (int q = 0; q < PTS; ++q) r[q] = r[q] > 0.0 ? sqrt_mid(r[q]) : 0.0;
    } else {
#pragma unroll
      for (int q = 0; q < PTS; ++q) r[q] = sqrt(r[q]);
    }
#pragma unroll
    for (int q = 0; q < PTS; ++q) {
      acc[q] += wj * pair_op<kSetGrad>(k, r[q], dx[q]);
      acc[PTS + q] += wj * pair_op<kSetGrad>(k, r[q], dy[q]);
    }
  }
  __shared__ double red[2 * PTS][kEvThreads / 64];
  block_sums(acc, red);
  if (threadIdx.x < 2 * PTS) {
    const int q = threadIdx.x % PTS, op = threadIdx.x < PTS ? RBFX_DX : RBFX_DY;
    const int64_t p = p0 + q;
    if (p >= npts) return;
    double s = 0.0;
    for (int w = 0; w < kEvThreads / 64; ++w) s += red[threadIdx.x][w];
    for (int64_t m = 0; m < M; ++m) {
      double o[RBFX_NOPS];
      mono_ops((int)m, px[p], py[p], o);
      s += coeffs[N + m] * o[op];
    }
    out[(int64_t)op * npts + p] = s;
  }
}

// Every operator of the mask (several, or a second derivative).
template <int KIND, bool FAST>
__global__ __launch_bounds__(kEvThreads) void eval_all_kernel(Kern k, int64_t N, int64_t M,
                                                              const double* __restrict__ cx,
                                                              const double* __restrict__ cy,
                                                              const double* __restrict__ coeffs,
                                                              int64_t npts, const double* __restrict__ px,
                                                              const double* __restrict__ py, uint32_t mask,
                                                              double* __restrict__ out) {
  pin_kind<KIND, FAST>(k);
  const int64_t p0 = (int64_t)blockIdx.x * kEvPts;
  double xp[kEvPts], yp[kEvPts];
  double acc[kEvPts][RBFX_NOPS];
#pragma unroll
  for (int q = 0; q < kEvPts; ++q) {
    const int64_t p = p0 + q < npts ? p0 + q : npts - 1;
    xp[q] = px[p];
    yp[q] = py[p];
#pragma unroll
    for (int t = 0; t < RBFX_NOPS; ++t) acc[q][t] = 0.0;
  }
  for (int64_t j = threadIdx.x; j < N; j += kEvThreads) {
    const double lam = coeffs[j];
    const double xj = cx[j], yj = cy[j];
#pragma unroll
    for (int q = 0; q < kEvPts; ++q) {
      double o[RBFX_NOPS];
      all_ops(k, xp[q] - xj, yp[q] - yj, o);
#pragma unroll
      for (int t = 0; t < RBFX_NOPS; ++t) acc[q][t] += lam * o[t];
    }
  }
  __shared__ double red[kEvPts][RBFX_NOPS][kEvThreads / 64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q < kEvPts; ++q) {
#pragma unroll
    for (int t = 0; t < RBFX_NOPS; ++t) {
      double v = acc[q][t];
      for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
      if (lane == 0) red[q][t][wid] = v;
    }
  }
  __syncthreads();
  if (threadIdx.x < kEvPts * RBFX_NOPS) {
    const int q = threadIdx.x / RBFX_NOPS, t = threadIdx.x % RBFX_NOPS;
    const int64_t p = p0 + q;
    if (p < npts && (mask & (1u << t))) {
      double s = 0.0;
      for (int w = 0; w < kEvThreads / 64; ++w) s += red[q][t][w];
      for (int64_t m = 0; m < M; ++m) {
        double o[RBFX_NOPS];
        mono_ops((int)m, xp[q], yp[q], o);
        s += coeffs[N + m] * o[t];
      }
      out[(int64_t)t * npts + p] = s;
    }
  }
}

// This thread's share of sum_i w_i op p_m(p_i).
__device__ inline double mono_share(int m, int64_t npts, const double* __restrict__ px, const double* __restrict__ py,
                                    int op, const double* __restrict__ w) {
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < npts; i += kEvThreads) {
    double o[RBFX_NOPS];
    mono_ops(m, px[i], py[i], o);
    acc += w[i] * o[op];
  }
  return acc;
}

// out[j] = sum_i w_i op phi(p_i, c_j), out[N+m] = sum_i w_i op p_m(p_i): a
// workgroup per monomial (first, they take longest), then one per PTS
// centres, its threads striding over the points.  0.45 ms for one component
// at 40,007 points and 10,000 centres; 3.5 ms when a workgroup took 64 centres
// and its four waves walked the points (157 workgroups, all seven operators
// of every pair).
template <int KIND, bool FAST, int SET, int PTS>
__global__ __launch_bounds__(kEvThreads) void eval_t_kernel(Kern k, int64_t N, int64_t M,
                                                            const double* __restrict__ cx,
                                                            const double* __restrict__ cy, int64_t npts,
                                                            const double* __restrict__ px,
                                                            const double* __restrict__ py, int op,
                                                            const double* __restrict__ w,
                                                            double* __restrict__ out) {
  pin_kind<KIND, FAST>(k);
  double acc[PTS];
#pragma unroll
  for (int q = 0; q < PTS; ++q) acc[q] = 0.0;
  __shared__ double red[PTS][kEvThreads / 64];
  const bool mono = (int64_t)blockIdx.x < M;
  const int64_t j0 = ((int64_t)blockIdx.x - M) * PTS;
  if (mono) {
    acc[0] = mono_share(blockIdx.x, npts, px, py, op, w);
  } else {
    double xj[PTS], yj[PTS];
#pragma unroll
    for (int q = 0; q < PTS; ++q) {
      const int64_t j = j0 + q < N ? j0 + q : N - 1;
      xj[q] = cx[j];
      yj[q] = cy[j];
    }
    if constexpr (SET != kSetAll) {
      pair_sums<SET, PTS, true>(k, npts, px, py, w, xj, yj, op == RBFX_DY, acc);
    } else {
      for (int64_t i = threadIdx.x; i < npts; i += kEvThreads) {
        const double wi = w[i], x = px[i], y = py[i];
#pragma unroll
        for (int q = 0; q < PTS; ++q) {
          double o[RBFX_NOPS];
          all_ops(k, x - xj[q], y - yj[q], o);
          acc[q] += wi * o[op];
        }
      }
    }
  }
  block_sums(acc, red);
  if (threadIdx.x >= (mono ? 1 : PTS)) return;
  const int64_t at = mono ? N + blockIdx.x : j0 + threadIdx.x;
  if (!mono && at >= N) return;
  out[at] = red[threadIdx.x][0] + red[threadIdx.x][1] + red[threadIdx.x][2] + red[threadIdx.x][3];
}

// The same for at most kChunkPoints points, each centre's sum in a fixed
// order: four quarters of the points, each summed in sequence, added in
// order.  The limit keeps results: the adjoint of implicit time stepping calls
// it at these sizes, where kappa ~ 1e10 turns another order of summation, no
// less accurate, into 2e-9 of its gradients (60 x 60 nodes, 8 steps).  A workgroup takes kChunkCentres centres: all its
// threads form the pairs of a tile (kChunkTile points of every quarter) in
// LDS while its first wave adds the tile before, a lane per (centre, quarter).
// 88 us for 3,480 points and 3,600 centres (r^3, value); 285 us when each lane
// formed and added its own pairs, 28 us for the whole-workgroup sums above.
constexpr int64_t kChunkPoints = 4096;
constexpr int kChunkCentres = 16, kChunkTile = 16;
template <int KIND, bool FAST, int SET>
__global__ __launch_bounds__(kEvThreads) void eval_t_chunk_kernel(Kern k, int64_t N, int64_t M,
                                                                  const double* __restrict__ cx,
                                                                  const double* __restrict__ cy, int64_t npts,
                                                                  const double* __restrict__ px,
                                                                  const double* __restrict__ py, int op,
                                                                  const double* __restrict__ w,
                                                                  double* __restrict__ out) {
  static_assert(kChunkCentres * kChunkTile == kEvThreads && 4 * kChunkCentres == 64, "a pair per thread and quarter");
  pin_kind<KIND, FAST>(k);
  constexpr int kQuarter = kChunkTile * kChunkCentres + 16;  // (the 16 keeps the quarters on distinct banks)
  __shared__ double pairs[2][4][kQuarter];
  __shared__ double wts[2][4][kChunkTile];
  __shared__ double red[4][kChunkCentres];
  const int tid = threadIdx.x;
  if ((int64_t)blockIdx.x < M) {
    const double acc[1] = {mono_share(blockIdx.x, npts, px, py, op, w)};
    block_sums(acc, red);
    if (tid == 0) out[N + blockIdx.x] = red[0][0] + red[0][1] + red[0][2] + red[0][3];
    return;
  }
  const int64_t j0 = ((int64_t)blockIdx.x - M) * kChunkCentres;
  const int ctr = tid % kChunkCentres, slot = tid / kChunkCentres;
  const int64_t j = j0 + ctr < N ? j0 + ctr : N - 1;
  const double xj = cx[j], yj = cy[j];
  const bool along_y = op == RBFX_DY;
  const int per = (int)((npts + 3) / 4);  // quarter q holds the points [q per, min((q + 1) per, npts))
  const int tiles = (per + kChunkTile - 1) / kChunkTile;
  auto pair = [&](double dx, double dy, double r) -> double {
    if constexpr (SET == kSetAll) {
      double o[RBFX_NOPS];
      all_ops(k, dx, dy, o);
      return o[op];
    } else {
      return pair_op<SET>(k, r, along_y ? dy : dx);
    }
  };
  double x[4], y[4], wq[4];
  auto load = [&](int t) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int at = t * kChunkTile + slot;
      const int64_t i = (int64_t)q * per + (at < per ? at : per - 1);
      const int64_t ii = i < npts ? i : npts - 1;  // (past a quarter's end: formed, not added)
      x[q] = px[ii];
      y[q] = py[ii];
      wq[q] = w[ii];
    }
  };
  double acc = 0.0;
  const int aq = tid / kChunkCentres;  // quarter that this lane of the first wave adds
  const int64_t left = npts - (int64_t)aq * per;
  const int mine = left < 0 ? 0 : left < per ? (int)left : per;
  auto add = [&](int t) {
    const int b = t & 1, n = mine - t * kChunkTile;
#pragma unroll
    for (int e = 0; e < kChunkTile; ++e) {
      const double v = __builtin_fma(wts[b][aq][e], pairs[b][aq][e * kChunkCentres + ctr], acc);
      acc = e < n ? v : acc;
    }
  };
  if (tiles > 0) load(0);
  for (int t = 0; t < tiles; ++t) {
    double dx[4], dy[4], r2[4];
    bool mid = true;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      dx[q] = x[q] - xj;
      dy[q] = y[q] - yj;
      r2[q] = dist2(dx[q], dy[q]);
      mid = mid && mid_or_zero(r2[q]);
    }
    const int b = t & 1;
    if (ctr == 0)
#pragma unroll
      for (int q = 0; q < 4; ++q) wts[b][q][slot] = wq[q];
    if (t + 1 < tiles) load(t + 1);
    if (__all(mid)) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        pairs[b][q][slot * kChunkCentres + ctr] = pair(dx[q], dy[q], r2[q] > 0.0 ? sqrt_mid(r2[q]) : 0.0);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) pairs[b][q][slot * kChunkCentres + ctr] = pair(dx[q], dy[q], sqrt(r2[q]));
    }
    // Tile t is whole; the other buffer was added before it is formed again.
    // (A plain barrier: __syncthreads() would wait for the next tile's loads.)
    __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (tid < 64) add(t);
  }
  if (tid < 64) red[aq][ctr] = acc;
  __syncthreads();
  if (tid < kChunkCentres && j0 + tid < N) out[j0 + tid] = red[0][tid] + red[1][tid] + red[2][tid] + red[3][tid];
}

// Four points (centres) per workgroup share its partners' loads; one where
// that would leave fewer than two workgroups per CU.  One value at 3,480
// points of 3,600 centres: 28 us with four, 29 us with one; at 33 points and
// 600 centres 18 us with four, 14 us with one.
static bool four_each(int64_t count) { return count >= 8 * (int64_t)device_info().num_cus; }

static int eval_launch(const Kern& k, int64_t N, int64_t M, const double* cx, const double* cy, const double* coeffs,
                       int64_t npts, const double* px, const double* py, uint32_t mask, double* out, hipStream_t s) {
  const int set = op_set(mask);
  int op = 0;
  while (!(mask & (1u << op))) ++op;
  const bool four = four_each(npts);
  const unsigned g4 = (unsigned)ceil_div(npts, kEvPts), g1 = (unsigned)npts;
#define RBFX_EVAL(SET_)                                                                                            \
  if (four)                                                                                                        \
    hipLaunchKernelGGL((eval_op_kernel<KIND_, FAST_, SET_, kEvPts>), dim3(g4), dim3(kEvThreads), 0, s, k, N, M, cx, \
                       cy, coeffs, npts, px, py, op, out);                                                         \
  else                                                                                                             \
    hipLaunchKernelGGL((eval_op_kernel<KIND_, FAST_, SET_, 1>), dim3(g1), dim3(kEvThreads), 0, s, k, N, M, cx, cy,  \
                       coeffs, npts, px, py, op, out)
  RBFX_KIND_SWITCH(k, {
    switch (set) {
      case kSetVal: RBFX_EVAL(kSetVal); break;
      case kSetGrad: RBFX_EVAL(kSetGrad); break;
      case kSetLap: RBFX_EVAL(kSetLap); break;
      case kSetBoth:
        if (four)
          hipLaunchKernelGGL((eval_grad_kernel<KIND_, FAST_, kEvPts>), dim3(g4), dim3(kEvThreads), 0, s, k, N, M, cx,
                             cy, coeffs, npts, px, py, out);
        else
          hipLaunchKernelGGL((eval_grad_kernel<KIND_, FAST_, 1>), dim3(g1), dim3(kEvThreads), 0, s, k, N, M, cx, cy,
                             coeffs, npts, px, py, out);
        break;
      default:
        hipLaunchKernelGGL((eval_all_kernel<KIND_, FAST_>), dim3(g4), dim3(kEvThreads), 0, s, k, N, M, cx, cy, coeffs,
                           npts, px, py, mask, out);
    }
  });
#undef RBFX_EVAL
  RBFX_CHECK_LAUNCH();
  return RBFX_OK;
}

static int eval_t_launch(const Kern& k, int64_t N, int64_t M, const double* cx, const double* cy, int64_t npts,
                         const double* px, const double* py, int op, const double* w, double* out, hipStream_t s) {
  const int set = op_set(1u << op);
  const bool chunks = npts <= kChunkPoints, four = four_each(N);
  const unsigned grid = (unsigned)(M + (chunks ? ceil_div(N, (int64_t)kChunkCentres) : four ? ceil_div(N, kEvPts) : N));
#define RBFX_EVAL_T(SET_)                                                                                        \
  if (chunks)                                                                                                    \
    hipLaunchKernelGGL((eval_t_chunk_kernel<KIND_, FAST_, SET_>), dim3(grid), dim3(kEvThreads), 0, s, k, N, M,   \
                       cx, cy, npts, px, py, op, w, out);                                                        \
  else if (four)                                                                                                 \
    hipLaunchKernelGGL((eval_t_kernel<KIND_, FAST_, SET_, kEvPts>), dim3(grid), dim3(kEvThreads), 0, s, k, N, M, \
                       cx, cy, npts, px, py, op, w, out);                                                        \
  else                                                                                                           \
    hipLaunchKernelGGL((eval_t_kernel<KIND_, FAST_, SET_, 1>), dim3(grid), dim3(kEvThreads), 0, s, k, N, M, cx,  \
                       cy, npts, px, py, op, w, out)
  RBFX_KIND_SWITCH(k, {
    switch (set) {
      case kSetVal: RBFX_EVAL_T(kSetVal); break;
      case kSetGrad: RBFX_EVAL_T(kSetGrad); break;
      case kSetLap: RBFX_EVAL_T(kSetLap); break;
      default: RBFX_EVAL_T(kSetAll);
    }
  });
#undef RBFX_EVAL_T
  RBFX_CHECK_LAUNCH();
  return RBFX_OK;
}

// q's rows without the terms: interior constant (+ row array), boundary
// values, zeros for the monomial rows.
__global__ __launch_bounds__(256) void rhs_init_kernel(int64_t N, int64_t M, int64_t Ni, double c0,
                                                      const double* __restrict__ crow,
                                                      const double* __restrict__ bc, double* __restrict__ q) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= N + M) return;
  double v = 0.0;
  if (i < Ni)
    v = c0 + (crow ? crow[i] : 0.0);
  else if (i < N)
    v = bc[i - Ni];
  q[i] = v;
}

// q[i] += w * row[i] * vals[i] over the interior rows.
__global__ __launch_bounds__(256) void rhs_accum_kernel(int64_t Ni, double w, const double* __restrict__ row,
                                                       const double* __restrict__ vals, double* __restrict__ q) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < Ni) q[i] += w * (row ? row[i] : 1.0) * vals[i];
}

}  // namespace rbfx

using namespace rbfx;

extern "C" int rbfx_eval(int kernel, double param, int64_t N, int64_t M, const double* d_cx,
                         const double* d_cy, const double* d_coeffs, int64_t npts,
                         const double* d_px, const double* d_py, uint32_t ops_mask, double* d_out,
                         void* stream) {
  RBFX_REQUIRE(kernel >= 0 && kernel <= 4, "unknown kernel %d", kernel);
  RBFX_REQUIRE(N > 0 && M >= 0 && M <= 15, "bad N / M");
  RBFX_REQUIRE(npts >= 0, "npts < 0");
  RBFX_REQUIRE(ops_mask != 0 && ops_mask < (1u << RBFX_NOPS), "bad ops_mask 0x%x", ops_mask);
  RBFX_REQUIRE(d_cx && d_cy && d_coeffs && d_out && (npts == 0 || (d_px && d_py)), "null pointer");
  if (npts == 0) return RBFX_OK;
  return eval_launch(make_kern(kernel, param), N, M, d_cx, d_cy, d_coeffs, npts, d_px, d_py, ops_mask, d_out,
                     as_stream(stream));
}

extern "C" int rbfx_eval_t(int kernel, double param, int64_t N, int64_t M, const double* d_cx,
                           const double* d_cy, int64_t npts, const double* d_px,
                           const double* d_py, int op, const double* d_w, double* d_out,
                           void* stream) {
  RBFX_REQUIRE(kernel >= 0 && kernel <= 4, "unknown kernel %d", kernel);
  RBFX_REQUIRE(N > 0 && M >= 0 && M <= 15, "bad N / M");
  RBFX_REQUIRE(op >= 0 && op < RBFX_NOPS, "bad op %d", op);
  RBFX_REQUIRE(npts >= 0, "npts < 0");
  RBFX_REQUIRE(d_cx && d_cy && d_w && d_out && (npts == 0 || (d_px && d_py)), "null pointer");
  return eval_t_launch(make_kern(kernel, param), N, M, d_cx, d_cy, npts, d_px, d_py, op, d_w, d_out,
                       as_stream(stream));
}

extern "C" size_t rbfx_rhs_workspace(const rbfx_problem* p) {
  if (!p || p->Ni < 0) return 0;
  return ws_round(sizeof(double) * (size_t)RBFX_NOPS * (size_t)p->Ni);
}

extern "C" int rbfx_rhs(const rbfx_problem* p, double constant, const double* d_const_row, int nterms,
                        const rbfx_rhs_term* terms, const double* d_bc, double* d_q, void* d_work,
                        size_t work_bytes, void* stream) {
  RBFX_REQUIRE(p != nullptr && d_q != nullptr, "null pointer");
  RBFX_REQUIRE(p->N > 0 && p->M >= 0 && p->M <= 15, "bad N / M");
  RBFX_REQUIRE(p->kernel >= 0 && p->kernel <= 4, "unknown kernel %d", p->kernel);
  RBFX_REQUIRE(p->Ni >= 0 && p->Nd >= 0 && p->Nn >= 0 && p->Nr >= 0 && p->Npd >= 0, "negative row-class size");
  RBFX_REQUIRE(p->Ni + p->Nd + p->Nn + p->Nr + 2 * p->Npd == p->N, "row classes do not add up to N");
  RBFX_REQUIRE(d_bc || p->N == p->Ni, "boundary values missing");
  RBFX_REQUIRE(nterms >= 0 && (nterms == 0 || terms), "bad terms");
  hipStream_t s = as_stream(stream);
  const int64_t N = p->N, M = p->M, Ni = p->Ni;
  hipLaunchKernelGGL(rhs_init_kernel, dim3((unsigned)ceil_div(N + M, 256)), dim3(256), 0, s, N, M, Ni, constant,
                     d_const_row, d_bc, d_q);
  RBFX_CHECK_LAUNCH();
  if (nterms == 0 || Ni == 0) return RBFX_OK;
  RBFX_REQUIRE(p->d_x && p->d_y, "node coordinates missing");
  Workspace ws(d_work, work_bytes);
  double* vals = ws.take<double>((size_t)RBFX_NOPS * (size_t)Ni);
  RBFX_REQUIRE(vals != nullptr, "rhs workspace too small");
  const Kern k = make_kern(p->kernel, p->param);
  for (int t = 0; t < nterms; ++t) {
    const rbfx_rhs_term& tm = terms[t];
    RBFX_REQUIRE(tm.op >= 0 && tm.op < RBFX_NOPS, "term %d: unknown operator %d", t, tm.op);
    RBFX_REQUIRE(tm.d_coeffs != nullptr, "term %d: coefficients missing", t);
    // the interior nodes are the first Ni nodes: evaluate op at them
    int st;
    if ((st = eval_launch(k, N, M, p->d_x, p->d_y, tm.d_coeffs, Ni, p->d_x, p->d_y, 1u << tm.op, vals, s))) return st;
    hipLaunchKernelGGL(rhs_accum_kernel, dim3((unsigned)ceil_div(Ni, 256)), dim3(256), 0, s, Ni, tm.weight,
                       tm.d_weight_row, vals + (size_t)tm.op * Ni, d_q);
    RBFX_CHECK_LAUNCH();
  }
  return RBFX_OK;
}
