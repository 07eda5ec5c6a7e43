// Device-side building blocks shared by the solve kernels (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rchol_amd {

// Control block in device memory.  The whole PCG state that the host would
// otherwise hold (alpha, beta, norms, counters) lives here so that an
// iteration never needs the host.
struct DevScalars {
  double bb;        // ||b||^2
  double rr;        // ||r||^2 of the recursively updated residual
  double rz;        // r.z of the current iteration
  double rz_old;    // r.z of the previous iteration (pcg.cpp:94 d2)
  double pr;        // p.r  (pcg.cpp:101)
  double pq;        // p.q  (pcg.cpp:102)
  double alpha;
  double beta;
  double tol;
  double relres;
  double qq;        // ||A x - b||^2 (final true residual)
  double rz_acc;    // r.z accumulated by the phases of a split backward sweep
  int k;            // completed iterations
  int maxit;
  int done;         // 1 once the loop test of pcg.cpp:82 fails
  int err;          // bit 0: a triangular-solve wait hit its bound
  int zero;         // constant 0: the stop flag of a standalone sweep
  int resid_period; // true-residual replacement period (0 = off)
  int strict;       // 1: grid reductions publish partials with release/acquire fences
  unsigned int ctr[8];  // last-block counters of the reductions (self-resetting)
  unsigned long long arrive;  // arrivals at the persistent sweeps' residency check
};

// ctr[CTR_CHUNK_Q] / [CTR_CHUNK_Q + 1]: chunk queue and exit count of the
// chunked sweeps (self-resetting)
enum { CTR_INIT = 0, CTR_BWD = 1, CTR_SPMVP = 2, CTR_UPD = 3, CTR_RES = 4, CTR_GEN = 5,
       CTR_CHUNK_Q = 6 };

// Sentinel bit patterns: signalling NaNs that arithmetic never produces.
constexpr unsigned long long kSent64 = 0x7FF4DEADBEEFCAFEull;
constexpr unsigned int kSent32 = 0x7FA5DEADu;

template <typename T> struct Sent;
template <> struct Sent<double> {
  static __device__ __forceinline__ double value() { return __longlong_as_double((long long)kSent64); }
  static __device__ __forceinline__ bool is(double v) {
    return (unsigned long long)__double_as_longlong(v) == kSent64;
  }
  static __device__ __forceinline__ double load_agent(const double *p) {
    unsigned long long b = __hip_atomic_load((const unsigned long long *)p, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
    return __longlong_as_double((long long)b);
  }
  static __device__ __forceinline__ void store_agent(double *p, double v) {
    __hip_atomic_store((unsigned long long *)p, (unsigned long long)__double_as_longlong(v),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
};
template <> struct Sent<float> {
  static __device__ __forceinline__ float value() { return __uint_as_float(kSent32); }
  static __device__ __forceinline__ bool is(float v) { return __float_as_uint(v) == kSent32; }
  static __device__ __forceinline__ float load_agent(const float *p) {
    unsigned int b = __hip_atomic_load((const unsigned int *)p, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
    return __uint_as_float(b);
  }
  static __device__ __forceinline__ void store_agent(float *p, float v) {
    __hip_atomic_store((unsigned int *)p, __float_as_uint(v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  }
};

// Loads of data that a kernel reads exactly once, non-temporal, so that the
// L2 keeps the gathered vector lines that neighbouring rows reuse instead of
// filling with the streamed matrix (K-column kernels, chunked sweeps).
#ifndef RCHOL_AMD_NT
#define RCHOL_AMD_NT 1
#endif
template <typename T>
__device__ __forceinline__ T ld_stream(const T *p) {
#if RCHOL_AMD_NT
  return __builtin_nontemporal_load(p);
#else
  return *p;
#endif
}
// The same as a choice of the kernel (the SpMV's stream form).
template <bool NT, typename T>
__device__ __forceinline__ T ld_once(const T *p) {
  if constexpr (NT) return __builtin_nontemporal_load(p);
  return *p;
}

// Bound on one dependency wait, in wall-clock ticks (the constant-rate
// counter runs at ~100 MHz: ~0.67 s), far beyond any legitimate wait.  A
// broken schedule therefore ends as an error flag, never as a hang; once the
// flag is up every other wait returns at its next check.
constexpr long long kWaitTicks = 1ll << 26;
// The bound every wait applies, per device (rchol_amd_set_option
// RCHOL_AMD_OPT_WAIT_TICKS lowers it to force the error path in tests).
__device__ long long g_wait_ticks = kWaitTicks;

// Back-off cap of the polling lane of await_batch, in s_sleep(1) units
// (64 clocks each): bounds the extra delay between publication and
// observation to ~kPollCap * 64 clocks.
#ifndef RCHOL_AMD_POLL_CAP
#define RCHOL_AMD_POLL_CAP 8
#endif
constexpr int kPollCap = RCHOL_AMD_POLL_CAP;

// The bound and back-off of one wait.
struct Poll {
  long long t0 = 0;
  int polls = 0, backoff = 1;
  // after a failed poll: every 8th time, whether the wait must end (past its
  // bound, or the error flag is up)
  __device__ __forceinline__ bool expired(const int *err) {
    if (polls == 0) t0 = wall_clock64();
    return (++polls & 7) == 0 &&
           (wall_clock64() - t0 > g_wait_ticks ||
            __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  }
  // doubling back-off up to cap units of 64 clocks
  __device__ __forceinline__ void sleep(int cap) {
    for (int i = 0; i < backoff; i++) __builtin_amdgcn_s_sleep(1);
    if (backoff < cap) backoff <<= 1;
  }
};

// Waits until *p is published (the same p in every active lane: one request
// per poll), with back-off and a bound that raises the error flag.
template <typename T>
__device__ __forceinline__ void await_value(const T *p, int *err) {
  Poll w;
  while (Sent<T>::is(Sent<T>::load_agent(p))) {
    if (w.expired(err)) {
      atomicOr(err, 1);
      break;
    }
    w.sleep(kPollCap);
  }
}

// Re-reads the pending slots of a round (j[u] < 0: an unused slot) and
// returns the lanes that still hold a sentinel.
template <typename T, int U>
__device__ __forceinline__ unsigned long long pending_lanes(const int (&j)[U], const T (&xv)[U]) {
  bool pend = false;
#pragma unroll
  for (int u = 0; u < U; u++) pend |= j[u] >= 0 && Sent<T>::is(xv[u]);
  return __ballot(pend);
}
template <typename T, int U>
__device__ __forceinline__ unsigned long long reread_pending(const T *x, const int (&j)[U],
                                                             T (&xv)[U], int stride = 1) {
#pragma unroll
  for (int u = 0; u < U; u++)
    if (j[u] >= 0 && Sent<T>::is(xv[u])) xv[u] = Sent<T>::load_agent(x + (size_t)j[u] * stride);
  return pending_lanes(j, xv);
}
template <typename T, int U>
__device__ __forceinline__ void zero_pending(const int (&j)[U], T (&xv)[U]) {
#pragma unroll
  for (int u = 0; u < U; u++)
    if (j[u] >= 0 && Sent<T>::is(xv[u])) xv[u] = T(0);
}

// Completes a round of U gathers per lane, xv[u] = x[j[u]] (j[u] < 0: an
// unused slot), once some lane of the wave still holds a sentinel.  Called
// by the whole wave, converged.  One lane polls the first pending address of
// the wave (a plain load may have hit a line cached before publication: then
// the first poll succeeds), and once that value is there every lane re-reads
// all of its pending slots at once, one load latency for the whole round.
// The slots are not re-read before that poll: most waits are long, and the
// re-reads of waves that are early load the fabric that the publications
// travel on.  A wait longer than g_wait_ticks raises the error flag; a raised
// flag zeroes what is still pending and returns.
// Slot u of a lane refers to x[j[u] * stride + col] (stride / col: the
// interleaved columns of a multi-right-hand-side block; 1 / 0 otherwise).
template <typename T, int U>
__device__ __forceinline__ void await_batch(const T *x, const int (&j)[U], T (&xv)[U], int *err,
                                            int stride = 1, int col = 0) {
  x += col;
  const int lane = __lane_id();
  for (unsigned long long mask = pending_lanes(j, xv); mask;) {
    const int leader = __ffsll((long long)mask) - 1;
    int jp = -1;
#pragma unroll
    for (int u = U - 1; u >= 0; u--)
      if (j[u] >= 0 && Sent<T>::is(xv[u])) jp = j[u];
    jp = __shfl(jp, leader, 64);
    if (lane == leader) await_value(x + (size_t)jp * stride, err);
    mask = reread_pending(x, j, xv, stride);
    if (mask && __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
      zero_pending(j, xv);
      break;
    }
  }
}

// Back-off cap of await_all, in s_sleep(1) units.
#ifndef RCHOL_AMD_POLL2_CAP
#define RCHOL_AMD_POLL2_CAP 1
#endif
constexpr int kPoll2Cap = RCHOL_AMD_POLL2_CAP;

// await_batch for a round whose proxy was published before it gathered: the
// latest levels are being computed, few entries are pending, and every lane
// re-reads its own each poll, so a value is seen one load after its
// publication instead of after a poll and a second, re-reading load.  Same
// bound, error flag and zeroing as await_batch.
template <typename T, int U>
__device__ __forceinline__ void await_all(const T *x, const int (&j)[U], T (&xv)[U], int *err) {
  Poll w;
  for (;;) {
    const unsigned long long mask = reread_pending(x, j, xv);
    if (!mask) return;
    if (w.expired(err)) {
      if (__lane_id() == __ffsll((long long)mask) - 1) atomicOr(err, 1);
      zero_pending(j, xv);
      return;
    }
    w.sleep(kPoll2Cap);
  }
}

// Sum over the L consecutive lanes of a row group (L a power of two <= 64),
// in every lane.  The steps pair lanes 1, 2, 4, 8, 16 and 32 apart (equal
// bits in both lanes of a pair, since the addition commutes): within 16 lanes
// by DPP moves -- once the lanes of a quad hold one value, the mirror of 8
// lanes is the exchange 4 apart, and the mirror of 16 the one 8 apart -- and
// across them by the lane swaps of gfx950.  No step goes through the LDS
// crossbar, which costs a wave that just saw its last value about 0.06 us per
// step (64 lanes, FP64: six steps of two words).
template <int CTRL>
__device__ __forceinline__ int dpp_word(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  return __int_as_float(dpp_word<CTRL>(__float_as_int(v)));
}
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
  return __hiloint2double(dpp_word<CTRL>(__double2hiint(v)), dpp_word<CTRL>(__double2loint(v)));
}
// v of this lane plus v of the lane 16 (32) apart.
__device__ __forceinline__ float add_16_apart(float v) {
  const auto w = __builtin_amdgcn_permlane16_swap(__float_as_int(v), __float_as_int(v), false, false);
  return __int_as_float(w[0]) + __int_as_float(w[1]);
}
__device__ __forceinline__ float add_32_apart(float v) {
  const auto w = __builtin_amdgcn_permlane32_swap(__float_as_int(v), __float_as_int(v), false, false);
  return __int_as_float(w[0]) + __int_as_float(w[1]);
}
__device__ __forceinline__ double add_16_apart(double v) {
  const int h = __double2hiint(v), l = __double2loint(v);
  const auto wh = __builtin_amdgcn_permlane16_swap(h, h, false, false);
  const auto wl = __builtin_amdgcn_permlane16_swap(l, l, false, false);
  return __hiloint2double(wh[0], wl[0]) + __hiloint2double(wh[1], wl[1]);
}
__device__ __forceinline__ double add_32_apart(double v) {
  const int h = __double2hiint(v), l = __double2loint(v);
  const auto wh = __builtin_amdgcn_permlane32_swap(h, h, false, false);
  const auto wl = __builtin_amdgcn_permlane32_swap(l, l, false, false);
  return __hiloint2double(wh[0], wl[0]) + __hiloint2double(wh[1], wl[1]);
}
template <int L, typename T>
__device__ __forceinline__ T group_sum(T v) {
  if (L >= 2) v += dpp_move<0xB1>(v);    // quad_perm [1, 0, 3, 2]
  if (L >= 4) v += dpp_move<0x4E>(v);    // quad_perm [2, 3, 0, 1]
  if (L >= 8) v += dpp_move<0x141>(v);   // mirror of 8 lanes
  if (L >= 16) v += dpp_move<0x140>(v);  // mirror of 16 lanes
  if (L >= 32) v = add_16_apart(v);
  if (L >= 64) v = add_32_apart(v);
  return v;
}

__device__ __forceinline__ double wave_sum(double v) { return group_sum<64>(v); }

// s / d with the reciprocal of d formed beforehand, so that a wave that just
// saw its last value is three dependent operations from its quotient instead
// of a whole division: q = s rd corrected by its exact remainder, which is
// s / d correctly rounded when rd is and nothing leaves the normal range
// (Markstein's theorem).  Anything else -- a pivot outside [2^-b, 2^b], a
// quotient that is zero, tiny, huge or not finite -- takes the division.
template <typename T>
struct QuotRange;
template <>
struct QuotRange<double> {
  static constexpr double lo = 0x1p-400, hi = 0x1p400;
};
template <>
struct QuotRange<float> {
  static constexpr float lo = 0x1p-40f, hi = 0x1p40f;
};
__device__ __forceinline__ double fma_of(double a, double b, double c) { return __fma_rn(a, b, c); }
__device__ __forceinline__ float fma_of(float a, float b, float c) { return __fmaf_rn(a, b, c); }
__device__ __forceinline__ double abs_of(double a) { return fabs(a); }
__device__ __forceinline__ float abs_of(float a) { return fabsf(a); }
template <typename T>
struct Divisor {
  T d, rd;
  bool plain;  // this lane divides
  __device__ __forceinline__ explicit Divisor(T d_) : d(d_), rd(T(1) / d_) {
    const T a = abs_of(rd);
    plain = !(a > QuotRange<T>::lo && a < QuotRange<T>::hi);
    asm volatile("" : "+v"(rd));  // formed here, before the waits
  }
  // s / d in the lanes that use it
  __device__ __forceinline__ T quotient(T s, bool used) const {
    const T q0 = s * rd;
    const T q = fma_of(fma_of(-q0, d, s), rd, q0);
    const T a = abs_of(q);
    const bool slow = plain || !(a > QuotRange<T>::lo && a < QuotRange<T>::hi);
    // a wave-uniform branch: otherwise the division is computed in every lane
    if (__ballot(used && slow)) return slow ? s / d : q;
    return q;
  }
};

// Block-wide sum of NV doubles (blockDim.x a multiple of 64, <= 1024);
// the result is valid in thread 0.  Deterministic for a fixed launch shape.
template <int NV>
__device__ __forceinline__ void block_sum(double (&v)[NV]) {
  __shared__ double red[NV][16];
#pragma unroll
  for (int i = 0; i < NV; i++) v[i] = wave_sum(v[i]);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if (lane == 0) {
#pragma unroll
    for (int i = 0; i < NV; i++) red[i][w] = v[i];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int i = 0; i < NV; i++) {
      double s = 0.0;
      for (int k = 0; k < nw; k++) s += red[i][k];
      v[i] = s;
    }
  }
  __syncthreads();
}

// Last-block reduction: every block publishes its NV partial sums and
// counts itself in; the block that arrives last sums all partials in block
// order (deterministic) and returns true with the totals in tot[] (thread 0
// only).  The counter resets itself, so the same kernel can be replayed from
// a captured graph.
//
// Publication.  strict == 1 is the textbook form: plain stores, then an
// acquire-release counter increment (an agent-scope release writes back the
// whole L2 of the XCD, once per block).  strict == 0 (default) keeps every
// byte of the handshake in agent-scope atomics instead: a partial is written
// by a value-returning exchange, the counter increment is issued only once
// every exchange has returned (an empty asm consumes the returned values),
// and the last block reads the partials with agent-scope atomic loads.  A
// returned read-modify-write has been performed at the point where every
// agent-scope atomic of every XCD is ordered, so the last block finds all
// partials there without any cache writeback.
template <int NV>
__device__ __forceinline__ bool grid_reduce(double (&v)[NV], double *partials, unsigned int *ctr,
                                            double (&tot)[NV], int strict) {
  block_sum<NV>(v);
  __shared__ int is_last;
  if (threadIdx.x == 0) {
    unsigned int prev;
    if (strict) {
#pragma unroll
      for (int i = 0; i < NV; i++) partials[(size_t)blockIdx.x * NV + i] = v[i];
      prev = __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    } else {
      unsigned long long got = 0;
#pragma unroll
      for (int i = 0; i < NV; i++)
        got ^= __hip_atomic_exchange(
            (unsigned long long *)(partials + (size_t)blockIdx.x * NV + i),
            (unsigned long long)__double_as_longlong(v[i]), __ATOMIC_RELAXED,
            __HIP_MEMORY_SCOPE_AGENT);
      asm volatile("" ::"v"(got) : "memory");
      prev = __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    is_last = (prev == gridDim.x - 1);
  }
  __syncthreads();
  if (!is_last) return false;
  if (strict) __atomic_thread_fence(__ATOMIC_ACQUIRE);
  double s[NV];
#pragma unroll
  for (int i = 0; i < NV; i++) s[i] = 0.0;
  for (unsigned int b = threadIdx.x; b < gridDim.x; b += blockDim.x) {
#pragma unroll
    for (int i = 0; i < NV; i++)
      s[i] += strict ? partials[(size_t)b * NV + i]
                     : Sent<double>::load_agent(partials + (size_t)b * NV + i);
  }
  block_sum<NV>(s);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int i = 0; i < NV; i++) tot[i] = s[i];
    __hip_atomic_store(ctr, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  return threadIdx.x == 0;
}

// Residency check of a persistent grid.  The level-scheduled sweeps can
// only finish when all of their workgroups are resident together (a wave
// may wait for a row of any other wave), so that is checked, not assumed:
//  * grid_arrive: every workgroup counts itself in at entry (one atomic, no
//    wait) and gets the count the whole grid reaches;
//  * wave_resident: every wave, before its first task that may wait for
//    another wave, waits (one polling lane, bounded) until that count is
//    reached.  Tasks that wait for nothing (level 0 of the forward sweep)
//    run first, while the rest of the grid is still being dispatched.
// A grid that does not fit -- too many workgroups, or CUs held by other
// work -- fails the bounded wait: the error flag gets bit 2 and the wave
// skips its tasks (taking part in the kernel's grid reduction all the same).
// The counter is never reset: each launch adds exactly gridDim.x arrivals,
// so the g-th launch of a grid waits for (g + 1) * gridDim.x; the host
// zeroes it whenever the grid size changes.
__device__ __forceinline__ unsigned long long grid_arrive(unsigned long long *arrive) {
  __shared__ unsigned long long target;
  if (threadIdx.x == 0) {
    const unsigned long long v =
        __hip_atomic_fetch_add(arrive, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    target = (v / gridDim.x + 1) * gridDim.x;
  }
  __syncthreads();
  return target;
}

__device__ __forceinline__ bool wave_resident(const unsigned long long *arrive,
                                              unsigned long long target, int *err) {
  int good = 1;
  if (__lane_id() == 0) {
    int backoff = 1;
    const long long t0 = wall_clock64();
    for (int polls = 1;
         __hip_atomic_load(arrive, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target;
         polls++) {
      for (int i = 0; i < backoff; i++) __builtin_amdgcn_s_sleep(1);
      if (backoff < 8) backoff <<= 1;
      if ((polls & 15) == 0 &&
          (wall_clock64() - t0 > g_wait_ticks ||
           __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
        atomicOr(err, 4);
        good = 0;
        break;
      }
    }
  }
  return __shfl(good, 0, 64) != 0;
}

}  // namespace rchol_amd
