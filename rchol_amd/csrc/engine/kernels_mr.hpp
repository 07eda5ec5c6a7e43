// Multi-right-hand-side kernels: K columns stored interleaved (row-major
// n x K, element (i, c) at i*K + c).  A lane owns one column (sweeps) or kCols
// neighbouring ones, so K or K / kCols lanes apply a matrix entry (index +
// value, loaded once) to K columns with one coalesced K-wide vector access.
// Every column runs its own PCG recurrence (pcg.cpp:57-127) with its own
// scalars and convergence mask; a converged column is frozen.
#pragma once
#include "kernels.hpp"

namespace rchol_amd {

constexpr int kMaxCols = 32;
// Workgroups of the K-column SpMV per CU, all resident (100^3, K = 32, with the
// p update: 6 per CU 593 us and spills, 5 495 us, 4 485 us).
#ifndef RCHOL_AMD_SPMV_MR_PER_CU
#define RCHOL_AMD_SPMV_MR_PER_CU 4
#endif
constexpr int kSpmvMrBlocksPerCu = RCHOL_AMD_SPMV_MR_PER_CU;
// Widest block whose sweeps take merged levels: a merged row is long, and K
// columns leave it 64 / K lanes per entry round.  Both sweeps of FP32 factors,
// plain -> merged: K = 4: 24^3 219 -> 101 us, 100^3 875 -> 621 us; K = 8: 217 ->
// 140 and 1018 -> 865; K = 16: 216 -> 218 and 1303 -> 1414; K = 32: 221 -> 366 and
// 1482 -> 2198.  (Wider kernels are compiled without them.)
constexpr int kMergeCols = 8;
// Columns per lane of the SpMV and the vector updates: a row takes half as many
// lanes as with one, so a wave holds twice as many rows (their index loads and
// gathers in flight) and its accesses are 16 bytes wide.
constexpr int kCols = 2;

// kCols neighbouring columns of one row, aligned as one element: the caller's
// blocks need no more.
template <typename T>
struct ColVec {
  typedef T type __attribute__((ext_vector_type(2), aligned(sizeof(T))));
};
template <typename T>
using Cols = typename ColVec<T>::type;
static_assert(kCols == 2, "ColVec");
template <typename T>
__device__ __forceinline__ Cols<T> ld_cols(const T *p) {
  return *(const Cols<T> *)p;
}
template <typename T>
__device__ __forceinline__ Cols<T> ld_cols_once(const T *p) {
  return __builtin_nontemporal_load((const Cols<T> *)p);
}
template <typename T>
__device__ __forceinline__ void st_cols(T *p, Cols<T> v) {
  *(Cols<T> *)p = v;
}
struct BatchScalars {
  double bb[kMaxCols], rr[kMaxCols], rz[kMaxCols], rz_old[kMaxCols];
  double pr[kMaxCols], pq[kMaxCols], alpha[kMaxCols], beta[kMaxCols];
  double relres[kMaxCols];
  int k[kMaxCols];
  int done[kMaxCols];
  int all_done;
  int ncols;  // live columns (<= K); padding columns start done
  int maxit;
  int err;
  int zero;
  int strict;  // 1: reductions publish partials with release/acquire fences
  double tol;
  unsigned int ctr[8];
  unsigned long long arrive;  // arrivals at the sweeps' residency check (grid_register)
};

// Sum lanes holding the same columns inside a wave (lanes l, l + P, l + 2P, ...).
template <int P>
__device__ __forceinline__ double column_sum(double v) {
#pragma unroll
  for (int off = P; off < 64; off <<= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// NV per-column block sums, then the last block sums every column over all
// blocks in block order (deterministic).  A lane brings C neighbouring
// columns, from C * (lane % (K / C)).  Returns true in every thread of the
// last block (block-uniform); threads c < K hold the totals of column c in tot.
// The publication handshake is grid_reduce's: value-returning atomic exchanges
// and a relaxed counter (strict == 0), or plain stores and an
// acquire-release counter (strict == 1).  All threads of the last block take
// the blocks' partials in turn, kPartsInFlight loads of each in flight, and
// the waves' sums are added in wave order: one thread per column walking
// every block is a chain of loads that the next kernel waits for (K = 4 at
// 48^3: SpMV 576 us with that chain, 77 us without).
constexpr int kPartsInFlight = 8;
template <int K, int C, int NV>
__device__ __forceinline__ bool column_grid_reduce(const double (&v)[NV][C], double *partials,
                                                   unsigned int *ctr, double (&tot)[NV],
                                                   int strict) {
  __shared__ double red[16][NV * K];
  __shared__ int is_last;
  constexpr int P = K / C, T = NV * K;  // slot t = i K + c: sum i of column c
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
  for (int i = 0; i < NV; i++)
#pragma unroll
    for (int k = 0; k < C; k++) {
      const double s = column_sum<P>(v[i][k]);
      if (lane < P) red[w][i * K + lane * C + k] = s;
    }
  __syncthreads();
  if (threadIdx.x < T) {
    double s = 0.0;
    for (int i = 0; i < nw; i++) s += red[i][threadIdx.x];
    double *slot = partials + (size_t)blockIdx.x * T + threadIdx.x;
    if (strict) {
      *slot = s;
    } else {
      const unsigned long long got = __hip_atomic_exchange(
          (unsigned long long *)slot, (unsigned long long)__double_as_longlong(s),
          __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      asm volatile("" ::"v"(got) : "memory");
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned int prev =
        strict ? __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT)
               : __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    is_last = (prev == gridDim.x - 1);
  }
  __syncthreads();
  if (!is_last) return false;
  if (strict) __atomic_thread_fence(__ATOMIC_ACQUIRE);
  // thread t: slot t % T of blocks t / T, t / T + blockDim / T, ...
  const unsigned int step = blockDim.x / T;
  double s = 0.0;
  for (unsigned int b0 = threadIdx.x / T; b0 < gridDim.x; b0 += step * kPartsInFlight) {
    double pv[kPartsInFlight];
#pragma unroll
    for (int u = 0; u < kPartsInFlight; u++) {
      const unsigned int b = b0 + u * step;
      const double *slot = partials + (size_t)b * T + threadIdx.x % T;
      pv[u] = b >= gridDim.x ? 0.0 : strict ? *slot : Sent<double>::load_agent(slot);
    }
#pragma unroll
    for (int u = 0; u < kPartsInFlight; u++) s += pv[u];
  }
  s = column_sum<T>(s);
  if (lane < T) red[w][lane] = s;
  __syncthreads();
  if (threadIdx.x < K)
#pragma unroll
    for (int i = 0; i < NV; i++) {
      tot[i] = 0.0;
      for (int k = 0; k < nw; k++) tot[i] += red[k][i * K + threadIdx.x];
    }
  __syncthreads();
  if (threadIdx.x == 0) __hip_atomic_store(ctr, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}
static_assert(2 * kMaxCols <= 64, "the slots of a block fit a wave");

// AND of the column masks into all_done (last block, after its column
// threads updated done[]).
template <int K>
__device__ __forceinline__ void set_all_done(BatchScalars *bs) {
  __syncthreads();
  if (threadIdx.x == 0) {
    int all = 1;
    for (int c = 0; c < K; c++) all &= bs->done[c];
    bs->all_done = all;
  }
}

// Level-scheduled sweep on K interleaved columns (the deadlock-freedom
// argument of k_sptrsv; per-wave task lists cut for K columns).  A row
// takes K * Le lanes: lane (grp, sub, c) = lane / (K Le), lane / K % Le,
// lane % K owns column c of entries sub, sub + Le, ... (from the row's end)
// of row grp of the pass, so one index/value load serves K columns and every
// gather is one contiguous K-wide segment.  A round issues kGather gathers per
// lane before looking at any; pending values are awaited wave-cooperatively.
// One column per lane, unlike the other kernels here: two double the registers
// that a wave holds while it waits, and the narrow levels, where a wave is one
// pass, get slower by what the wide ones gain and more (100^3 FP32, K = 32:
// 0.74 -> 1.11 ms forward; K = 4: 0.47 -> 0.57).
// FUSE 1: sentinel into aux; FUSE 2: per-column dotv.x -> rz, beta.
// merged: the row may also hold right-hand sides of its own level group
// (column t stored as -2 - t), as in row_dot.
template <typename VT, typename XT, typename BT, int Le, int K>
__device__ __forceinline__ XT row_dot_mr(int e0, int e1, int sub, int c,
                                         const int *__restrict__ ci, const VT *__restrict__ cv,
                                         const XT *x, const BT *__restrict__ rhs, int *err,
                                         bool merged) {
  XT acc = 0;
  constexpr int kRound = kGather * Le;
  for (int r = (e1 - e0 + kRound - 1) / kRound - 1; r >= 0; r--) {  // oldest first, as in row_dot
    const int last = e1 - 1 - sub - r * kRound;
    int j[kGather];
    VT v[kGather];
    XT xv[kGather];
#pragma unroll
    for (int u = 0; u < kGather; u++) {
      const int e = last - u * Le;
      j[u] = e >= e0 ? ci[e] : -1;
      v[u] = e >= e0 ? cv[e] : VT(0);
    }
#pragma unroll
    for (int u = 0; u < kGather; u++) xv[u] = j[u] < 0 ? XT(0) : x[(size_t)j[u] * K + c];
    if (K <= kMergeCols && merged) {
      BT bv[kGather];
#pragma unroll
      for (int u = 0; u < kGather; u++)
        bv[u] = j[u] < -1 ? rhs[(size_t)(-2 - j[u]) * K + c] : (BT)0;
#pragma unroll
      for (int u = 0; u < kGather; u++)
        if (j[u] < -1) xv[u] = (XT)bv[u];
    }
    if (pending_lanes(j, xv)) await_batch<XT, kGather>(x, j, xv, err, K, c);
#pragma unroll
    for (int u = 0; u < kGather; u++) acc += (XT)v[u] * xv[u];
  }
  return acc;
}

template <typename VT, typename XT, typename BT, int K, int Le, int FUSE>
__device__ __forceinline__ void sweep_task_mr(int cnt, int m_row, int m_e0, int m_e1, VT m_dg,
                                              const int *__restrict__ ci,
                                              const VT *__restrict__ cv,
                                              const BT *__restrict__ rhs, XT *x,
                                              XT *__restrict__ aux,
                                              const double *__restrict__ dotv, int *err,
                                              double &dacc, bool merged) {
  constexpr int W = K * Le, R = 64 / W;
  const int lane = threadIdx.x & 63;
  const int c = lane % K, sub = (lane / K) % Le, grp = lane / W;
  for (int base = 0; base < cnt; base += R) {
    const int k = base + grp;  // < 64
    const int row = __shfl(m_row, k, 64);
    int e0 = __shfl(m_e0, k, 64), e1 = __shfl(m_e1, k, 64);
    const VT dg = __shfl(m_dg, k, 64);
    const bool live = k < cnt;
    if (!live) e1 = e0;
    const size_t o = (size_t)row * K + c;
    // before the waits: what the epilogue needs besides the sum
    const BT b = (live && sub == 0) ? rhs[o] : (BT)0;
    const double dv = FUSE == 2 && live && sub == 0 ? dotv[o] : 0.0;
    XT acc = row_dot_mr<VT, XT, BT, Le, K>(e0, e1, sub, c, ci, cv, x, rhs, err, merged);
#pragma unroll
    for (int off = K; off < W; off <<= 1) acc += __shfl_xor(acc, off, 64);
    if (live && sub == 0) {
      const XT v = ((XT)b - acc) / (XT)dg;
      Sent<XT>::store_agent(x + o, v);
      if (FUSE == 1) aux[o] = Sent<XT>::value();
      if (FUSE == 2) dacc += dv * (double)v;
    }
  }
}

template <typename VT, typename XT, typename BT, int K, int FUSE>
__global__ __launch_bounds__(256) void k_sptrsv_mr(
    const int *__restrict__ wave_ptr, const SweepTask *__restrict__ wt,
    const int *__restrict__ slot_row,
    const int *__restrict__ rp, const int *__restrict__ ci, const VT *__restrict__ cv,
    const int *__restrict__ mrp, const int *__restrict__ mci, const VT *__restrict__ mcv,
    const VT *__restrict__ diag, const BT *__restrict__ rhs, XT *x, XT *__restrict__ aux,
    const double *__restrict__ dotv, double *__restrict__ partials, BatchScalars *bs,
    const int *stop) {
  if (*stop) return;
  const int lane = threadIdx.x & 63;
  const int wave = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  int *err = &bs->err;
  double dacc[1][1] = {{0.0}};
  const unsigned long long arrivals = grid_arrive(&bs->arrive);
  const int k1 = wave_ptr[wave + 1];
  int k = wave_resident(&bs->arrive, arrivals, err) ? wave_ptr[wave] : k1;
  int n_info = 0, n_row = 0, n_e0 = 0, n_e1 = 0;
  VT n_dg = 1;
  auto fetch = [&](int kk) {
    const int s = wt[kk].s0;
    n_info = wt[kk].info;
    if (lane < (n_info & ((1 << kTaskInfoShift) - 1))) {
      const int *rq = K <= kMergeCols && (n_info & kTaskMerged) ? mrp : rp;
      n_row = slot_row[s + lane];
      n_e0 = rq[s + lane];
      n_e1 = rq[s + lane + 1];
      n_dg = diag[s + lane];
    }
  };
  if (k < k1) fetch(k);
  for (; k < k1; k++) {
    const int info = n_info;
    const int lg = (info >> kTaskInfoShift) & 15;
    const bool merged = K <= kMergeCols && (info & kTaskMerged) != 0;
    const int cnt = info & ((1 << kTaskInfoShift) - 1);
    const int m_row = n_row, m_e0 = n_e0, m_e1 = n_e1;
    const VT m_dg = n_dg;
    if (k + 1 < k1) fetch(k + 1);
#define RCHOL_MR_TASK(LE)                                                                  \
  sweep_task_mr<VT, XT, BT, K, ((LE) * K <= 64 ? (LE) : 64 / K), FUSE>(                    \
      cnt, m_row, m_e0, m_e1, m_dg, merged ? mci : ci, merged ? mcv : cv, rhs, x, aux, dotv, \
      err, dacc[0][0], merged)
    switch (lg) {
      case 0: RCHOL_MR_TASK(1); break;
      case 1: RCHOL_MR_TASK(2); break;
      case 2: RCHOL_MR_TASK(4); break;
      case 3: RCHOL_MR_TASK(8); break;
      default: RCHOL_MR_TASK(16); break;
    }
#undef RCHOL_MR_TASK
  }
  if (FUSE == 2) {
    double tot[1];
    if (column_grid_reduce<K, 1, 1>(dacc, partials, &bs->ctr[CTR_BWD], tot, bs->strict) &&
        threadIdx.x < K) {
      const int cc = threadIdx.x;
      bs->rz[cc] = tot[0];
      bs->beta[cc] = (bs->k[cc] > 0) ? tot[0] / bs->rz_old[cc] : 0.0;
      bs->rz_old[cc] = tot[0];
    }
  }
}

// r = b, x = 0 (or keep), y = sentinel, per-column ||b||^2 and loop test.
template <typename YT, int K>
__global__ __launch_bounds__(256) void k_init_mr(int n, const double *__restrict__ b, double *r,
                                                 double *x, int keep_x, YT *y, double *partials,
                                                 BatchScalars *bs) {
  double acc[1][1] = {{0.0}};
  const size_t total = (size_t)n * K;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (size_t)gridDim.x * blockDim.x) {
    const double bi = b[i];
    r[i] = bi;
    if (!keep_x) x[i] = 0.0;
    y[i] = Sent<YT>::value();
    acc[0][0] += bi * bi;
  }
  double tot[1];
  if (column_grid_reduce<K, 1, 1>(acc, partials, &bs->ctr[CTR_INIT], tot, bs->strict)) {
    if (threadIdx.x < K) {
      const int cc = threadIdx.x;
      bs->bb[cc] = tot[0];
      bs->rr[cc] = tot[0];
      bs->k[cc] = 0;
      bs->beta[cc] = 0.0;
      bs->alpha[cc] = 0.0;
      bs->done[cc] = (cc >= bs->ncols) || !(sqrt(tot[0]) > sqrt(tot[0]) * bs->tol && 0 < bs->maxit);
    }
    if (threadIdx.x == 0) bs->err = 0;
    set_all_done<K>(bs);
  }
}

// Rows of a multi-column SpMV: K / kCols lanes per row (lane p = columns
// kCols p, ...), the XCD-contiguous walk of xcd_rows in steps of the wave's
// rows.  Entries go in rounds of kGather per lane: all index/value
// loads, then all K-wide gathers, then the products.
template <int K>
__device__ __forceinline__ RowWalk xcd_rows_mr(int n) {
  constexpr int P = K / kCols, R = 64 / P;
  const int X = (gridDim.x % 8 == 0) ? 8 : 1;
  const int x = blockIdx.x % X, jb = blockIdx.x / X, nbx = gridDim.x / X;
  const int wpb = blockDim.x >> 6;
  const int lo = (int)((long long)n * x / X);
  RowWalk w;
  w.hi = (int)((long long)n * (x + 1) / X);
  w.first = lo + (jb * wpb + (threadIdx.x >> 6)) * R + (threadIdx.x & 63) / P;
  w.step = nbx * wpb * R;
  return w;
}

template <int K>
__device__ __forceinline__ Cols<double> row_dot_a(int e0, int e1, const int *__restrict__ ci,
                                                  const double *__restrict__ av, const double *g,
                                                  int col) {
  Cols<double> acc = Cols<double>(0.0);
  for (int b0 = e0; b0 < e1; b0 += kGather) {
    int j[kGather];
    double a[kGather];
    Cols<double> pv[kGather];
#pragma unroll
    for (int u = 0; u < kGather; u++) {
      const int e = b0 + u;
      j[u] = e < e1 ? ld_stream(ci + e) : -1;
      a[u] = e < e1 ? ld_stream(av + e) : 0.0;
    }
#pragma unroll
    for (int u = 0; u < kGather; u++)
      pv[u] = j[u] >= 0 ? ld_cols(g + (size_t)j[u] * K + col) : Cols<double>(0.0);
#pragma unroll
    for (int u = 0; u < kGather; u++) {
      acc[0] += a[u] * pv[u][0];
      acc[1] += a[u] * pv[u][1];
    }
  }
  return acc;
}

// p_new = z + beta_c p_old (p = z at k_c == 0), ahead of the SpMV that gathers
// it: formed on the fly, every one of a row's entries would gather z and
// p_old instead of p.
template <typename ZT, int K>
__global__ __launch_bounds__(256) void k_p_update_mr(int n, const ZT *__restrict__ z,
                                                     const double *__restrict__ p_old,
                                                     double *__restrict__ p_new,
                                                     const BatchScalars *bs) {
  if (bs->all_done) return;
  const int col = threadIdx.x % (K / kCols) * kCols;
  const bool f0 = bs->k[col] == 0, f1 = bs->k[col + 1] == 0;
  const double b0 = bs->beta[col], b1 = bs->beta[col + 1];
  const size_t total = (size_t)n * K;
  const size_t step = (size_t)gridDim.x * blockDim.x * kCols;
  for (size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * kCols; i < total; i += step) {
    const Cols<ZT> zi = ld_cols(z + i);
    const Cols<double> po = ld_cols_once(p_old + i);
    Cols<double> pn;
    pn[0] = f0 ? (double)zi[0] : b0 * po[0] + (double)zi[0];
    pn[1] = f1 ? (double)zi[1] : b1 * po[1] + (double)zi[1];
    st_cols(p_new + i, pn);
  }
}

// q = A p, per-column p.r and p.q -> alpha_c.  Bound by the K-wide gathers of p
// that leave the XCDs' L2 (256^3, K = 32: 35.1 GB in 6.0 ms, 5.8 TB/s, for 14.4 GB
// of arrays).  100^3, K = 32, FP32 factor: p update and SpMV 405 us, 1408 us
// before, when one lane per column gathered z and p_old for every entry and one
// thread per column walked the blocks' partials.
template <int K>
__global__ __launch_bounds__(256, kSpmvMrBlocksPerCu) void k_spmv_p_mr(
    int n, const int *__restrict__ rp, const int *__restrict__ ci, const double *__restrict__ av,
    const double *__restrict__ p, double *__restrict__ q, const double *__restrict__ r,
    double *partials, BatchScalars *bs) {
  if (bs->all_done) return;
  const int col = threadIdx.x % (K / kCols) * kCols;
  const RowWalk rw = xcd_rows_mr<K>(n);
  double dots[2][kCols] = {{0.0, 0.0}, {0.0, 0.0}};  // p.r, p.q
  for (int row = rw.first; row < rw.hi; row += rw.step) {
    const int e0 = ld_stream(rp + row), e1 = ld_stream(rp + row + 1);
    const size_t o = (size_t)row * K + col;
    const Cols<double> pi = ld_cols(p + o), ri = ld_cols_once(r + o);
    const Cols<double> acc = row_dot_a<K>(e0, e1, ci, av, p, col);
    st_cols(q + o, acc);
    for (int i = 0; i < kCols; i++) {
      dots[0][i] += pi[i] * ri[i];
      dots[1][i] += pi[i] * acc[i];
    }
  }
  double tot[2];
  if (column_grid_reduce<K, kCols, 2>(dots, partials, &bs->ctr[CTR_SPMVP], tot, bs->strict) &&
      threadIdx.x < K) {
    const int cc = threadIdx.x;
    bs->pr[cc] = tot[0];
    bs->pq[cc] = tot[1];
    bs->alpha[cc] = tot[0] / tot[1];
  }
}

// x += alpha_c p, r -= alpha_c q for live columns; ||r_c||^2; y = sentinel;
// the last block advances k_c and re-evaluates every column's loop test.
// Memory-bound: 1.66 GB at 100^3, K = 32 take 335 us (4.9 TB/s); 552 us before
// with one column per lane and the serial tail.
template <typename YT, int K>
__global__ __launch_bounds__(256) void k_update_mr(int n, const double *__restrict__ p,
                                                   const double *__restrict__ q, double *x,
                                                   double *r, YT *y, double *partials,
                                                   BatchScalars *bs) {
  if (bs->all_done) return;
  const int col = threadIdx.x % (K / kCols) * kCols;
  const bool l0 = !bs->done[col], l1 = !bs->done[col + 1];
  const double a0 = bs->alpha[col], a1 = bs->alpha[col + 1];
  double acc[1][kCols] = {{0.0, 0.0}};
  const size_t total = (size_t)n * K;
  const size_t step = (size_t)gridDim.x * blockDim.x * kCols;
  for (size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * kCols; i < total; i += step) {
    Cols<double> ri = ld_cols(r + i);
    if (l0 || l1) {
      const Cols<double> pi = ld_cols(p + i), qi = ld_cols_once(q + i);
      Cols<double> xi = ld_cols(x + i);
      if (l0) {
        xi[0] += a0 * pi[0];
        ri[0] = ri[0] - a0 * qi[0];
      }
      if (l1) {
        xi[1] += a1 * pi[1];
        ri[1] = ri[1] - a1 * qi[1];
      }
      st_cols(x + i, xi);
      st_cols(r + i, ri);
    }
    st_cols(y + i, Cols<YT>(Sent<YT>::value()));
    acc[0][0] += ri[0] * ri[0];
    acc[0][1] += ri[1] * ri[1];
  }
  double tot[1];
  if (column_grid_reduce<K, kCols, 1>(acc, partials, &bs->ctr[CTR_UPD], tot, bs->strict)) {
    if (threadIdx.x < K) {
      const int cc = threadIdx.x;
      if (!bs->done[cc]) {
        const int k = bs->k[cc] + 1;
        bs->k[cc] = k;
        bs->rr[cc] = tot[0];
        bs->done[cc] = !(sqrt(tot[0]) > sqrt(bs->bb[cc]) * bs->tol && k < bs->maxit);
      }
    }
    set_all_done<K>(bs);
  }
}

// Per-column true residual ||A x - b|| / ||b|| (pcg.cpp:116-118); with
// bvec == null a plain Y = A X.
template <int K>
__global__ __launch_bounds__(256, kSpmvMrBlocksPerCu) void k_spmv_res_mr(
    int n, const int *__restrict__ rp, const int *__restrict__ ci, const double *__restrict__ av,
    const double *__restrict__ x, const double *__restrict__ bvec, double *__restrict__ y,
    double *partials, BatchScalars *bs) {
  const int col = threadIdx.x % (K / kCols) * kCols;
  const RowWalk rw = xcd_rows_mr<K>(n);
  double aqq[1][kCols] = {{0.0, 0.0}};
  for (int row = rw.first; row < rw.hi; row += rw.step) {
    const int e0 = ld_stream(rp + row), e1 = ld_stream(rp + row + 1);
    const size_t o = (size_t)row * K + col;
    const Cols<double> bi = bvec ? ld_cols(bvec + o) : Cols<double>(0.0);
    Cols<double> acc = row_dot_a<K>(e0, e1, ci, av, x, col);
    for (int i = 0; i < kCols; i++) {
      acc[i] -= bi[i];
      aqq[0][i] += acc[i] * acc[i];
    }
    st_cols(y + o, acc);
  }
  if (bvec) {
    double tot[1];
    if (column_grid_reduce<K, kCols, 1>(aqq, partials, &bs->ctr[CTR_RES], tot, bs->strict) &&
        threadIdx.x < K)
      bs->relres[threadIdx.x] = sqrt(tot[0]) / sqrt(bs->bb[threadIdx.x]);
  }
}

}  // namespace rchol_amd
