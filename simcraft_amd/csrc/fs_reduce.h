// fs_reduce.h - fixed-order reductions and ready-flag exchange shared by the pressure solvers
// (fs_pcg.hip, fs_mg.hip). Every reduction adds in one fixed tree, so results do not depend on
// scheduling and a CPU restatement of the tree reproduces them bit for bit.
#pragma once
#include "fs_ctx.h"

namespace {

constexpr long SPIN_LIMIT = 1000000;  // bounded wait (~1 s), then the solve reports a device error
enum { STOP_RUN = 0, STOP_CONVERGED = 1, STOP_ABORT = 2 };

// ---- fixed-tree reductions -------------------------------------------------------------------
__device__ inline double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = v + __shfl_xor(v, off, 64);
  return v;
}
__device__ inline double wave_max(double v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    double o = __shfl_xor(v, off, 64);
    v = (v < o) ? o : v;
  }
  return v;
}
// Per-thread values of a block's first 256 threads -> (w0 + w1) + (w2 + w3) of wave butterflies
// (the other threads of a larger block only take part in the barriers).
__device__ inline double block_sum256(double v, double* sm) {
  double w = wave_sum(v);
  int wid = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0 && wid < 4) sm[wid] = w;
  __syncthreads();
  double r = (sm[0] + sm[1]) + (sm[2] + sm[3]);
  __syncthreads();
  return r;
}
__device__ inline double block_max256(double v, double* sm) {
  double w = wave_max(v);
  int wid = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0 && wid < 4) sm[wid] = w;
  __syncthreads();
  double r = sm[0];
  for (int q = 1; q < 4; q++) r = (r < sm[q]) ? sm[q] : r;
  __syncthreads();
  return r;
}
// ---- boundary exchange between bricks ---------------------------------------------------------
// A brick hands its boundary row to the next brick through a small exchange array. Every entry
// holds a sentinel until the producer stores the value with an agent-scope atomic store; the
// consumer polls the entry with agent-scope atomic loads until the sentinel is gone, uses the
// value and stores the sentinel back. The sentinel is a signalling-NaN bit pattern, which
// floating-point arithmetic never returns, so every exchanged value is its own ready flag and
// no fence or cache maintenance is needed. Polls are bounded: after SPIN_LIMIT the wave gives
// up, counts a timeout and the host reports FS_DEVICE_ERROR.
constexpr unsigned long long XSENT = 0x7FF4DEADBEEF0001ull;

__device__ inline double xload(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void xstore(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline bool xready(double v) { return (unsigned long long)__double_as_longlong(v) != XSENT; }
__device__ inline double xsent() { return __longlong_as_double((long long)XSENT); }

// Wait until *p holds a written value; false when the wait gave up (the solve then reports
// FS_DEVICE_ERROR and every other waiter gives up within 256 polls).
__device__ inline bool xwait(const double* p, PcgScalars* sc) {
  long spins = 0;
  while (!xready(xload(p))) {
    __builtin_amdgcn_s_sleep(1);
    if ((++spins & 255) == 0) {
      int to = __hip_atomic_load(&sc->wait_timeouts, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (to != 0 || spins > SPIN_LIMIT) {
        atomicAdd(&sc->wait_timeouts, 1);
        return false;
      }
    }
  }
  return true;
}

__device__ inline double xpoll(const double* p, double v, PcgScalars* sc) {
  long spins = 0;
  while (!xready(v)) {
    __builtin_amdgcn_s_sleep(1);
    v = xload(p);
    if ((++spins & 255) == 0) {
      int to = __hip_atomic_load(&sc->wait_timeouts, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (to != 0 || spins > SPIN_LIMIT) {
        atomicAdd(&sc->wait_timeouts, 1);
        return 0.0;  // give up: results are invalid and the solve reports FS_DEVICE_ERROR
      }
    }
  }
  return v;
}

// High word of the sentinel. Arithmetic never returns a signalling NaN, so for computed values
// the high word alone identifies the sentinel.
constexpr uint32_t XSENT_HI = (uint32_t)(XSENT >> 32);
__device__ __forceinline__ bool xunset(double v) { return (uint32_t)__double2hiint(v) == XSENT_HI; }

// ---- cross-block reductions --------------------------------------------------------------------
// Every block (in the sweeps: every brick) stores its partials with agent-scope atomic stores into
// entries that otherwise hold the sentinel, so a stored partial is its own ready flag and no
// fence is needed: an agent-scope fence writes back and invalidates the L2 on this GPU, which,
// done by every block, costs more than the kernel's own work. The block dispatched last (the
// brick with the last ticket) waits until every entry is set, reduces them in the fixed order and
// stores the sentinel back, so the entries are unset again for the next kernel.

// Sum of the terms done(e, load(e)) of a chunk's elements e = 0 .. 4095 with live(e) (0 for the others)
// in the fixed order of 256 threads with 16 elements each (thread t: e = t + 256 m, m ascending), by TH
// threads; the value is that of the first 256 threads. With TH = 1024, thread (g, t) = (tid / 256,
// tid % 256) evaluates m = 4g .. 4g + 3 and the terms meet in LDS (TERMS<1024> doubles): the choice
// where a kernel has too few chunks to hide a thread's sixteen elements in turn by other blocks. There
// G of the four at a time are loaded before any is stored, unless none of the wave's is live: so load
// only reads, any element, and done writes.
template <int TH>
constexpr int CHUNK_TERMS = TH == 256 ? 1 : 4096;
template <int TH, class V, int G, class A, class L, class D>
__device__ __forceinline__ double chunk_sum(double* terms, A&& live, L&& load, D&& done) {
  double a = 0.0;
  if constexpr (TH == 256) {
#pragma unroll 1
    for (int m = 0; m < 16; m++) {
      const int e = 256 * m + (int)threadIdx.x;
      a += live(e) ? done(e, load(e)) : 0.0;
    }
  } else {
    static_assert(TH == 1024, "four groups of 256 threads");
    const int e0 = 1024 * (int)(threadIdx.x >> 8) + (int)(threadIdx.x & 255);
    bool on[4];
#pragma unroll
    for (int q = 0; q < 4; q++) on[q] = live(e0 + 256 * q);
    double term[4] = {0.0, 0.0, 0.0, 0.0};
    if (__builtin_amdgcn_ballot_w64(on[0] || on[1] || on[2] || on[3])) {
#pragma unroll
      for (int q0 = 0; q0 < 4; q0 += G) {
        V v[G];
#pragma unroll
        for (int q = 0; q < G; q++) v[q] = load(e0 + 256 * (q0 + q));
#pragma unroll
        for (int q = 0; q < G; q++)
          if (on[q0 + q]) term[q0 + q] = done(e0 + 256 * (q0 + q), v[q]);
      }
    }
#pragma unroll
    for (int q = 0; q < 4; q++) terms[e0 + 256 * q] = term[q];
    __syncthreads();
    if (threadIdx.x < 256) {
#pragma unroll
      for (int m = 0; m < 16; m++) a += terms[256 * m + threadIdx.x];
    }
  }
  return a;
}
// The maximum over a block's threads t, t + 256, .. to thread t of the first 256 (order-free).
template <int TH>
__device__ __forceinline__ double chunk_max(double mx, double* terms) {
  if constexpr (TH > 256) {
    __syncthreads();
    terms[threadIdx.x] = mx;
    __syncthreads();
    if (threadIdx.x < 256)
      for (int g = 1; g < TH / 256; g++) {
        const double o = terms[256 * g + threadIdx.x];
        mx = (mx < o) ? o : mx;
      }
  }
  return mx;
}

// The last block reads each entry as it waits for it, and keeps the value: a pass that only waits
// and another that reads again is one more round trip to memory at the end of every kernel that
// reduces, and nothing else runs by then (us, two passes / one: FP64 SpMV 13.6 / 12.0 at 32^3, forward
// sweep 17.1 / 16.3; mixed multigrid's update with two arrays 8.0 / 7.4 at 64^3, 41.1 / 34.8 at 256^3,
// 4096 entries). An entry is returned to the sentinel by the thread that read it. A wait that gives
// up yields 0 and counts a timeout (the solve then reports FS_DEVICE_ERROR).

// Fixed tree over the n entries of p (thread t < 256 sums p[t + 256 m] for m ascending, then
// block_sum256) and, where p2 is given, the maximum over p2 (order-free: the comparison never takes
// a NaN). All threads of the block call.
struct GatherSumMax {
  double sum, max;
};
__device__ inline GatherSumMax gather256(double* p, double* p2, int n, double* sm, PcgScalars* sc) {
  constexpr int K = 4;  // entries in flight per thread and array
  double a = 0.0, mx = 0.0;
  if (threadIdx.x < 256) {
    for (int m0 = threadIdx.x; m0 < n; m0 += 256 * K) {
      double v[K], w[K];
#pragma unroll
      for (int q = 0; q < K; q++) {
        const int m = m0 + 256 * q;
        v[q] = m < n ? xload(p + m) : 0.0;
        w[q] = p2 && m < n ? xload(p2 + m) : 0.0;
      }
#pragma unroll
      for (int q = 0; q < K; q++) {
        const int m = m0 + 256 * q;
        if (m >= n) continue;
        a += xpoll(p + m, v[q], sc);
        xstore(p + m, xsent());
        if (p2) {
          const double x = xpoll(p2 + m, w[q], sc);
          mx = (mx < x) ? x : mx;
          xstore(p2 + m, xsent());
        }
      }
    }
  }
  GatherSumMax r;
  r.sum = block_sum256(a, sm);
  r.max = p2 ? block_max256(mx, sm) : 0.0;
  return r;
}
// The same by one 64-lane wave (lane l plays threads l, l + 64, l + 128, l + 192).
__device__ inline GatherSumMax gather_wave(double* p, double* p2, int n, PcgScalars* sc) {
  const int lane = threadIdx.x & 63;
  double w[4] = {0.0, 0.0, 0.0, 0.0}, mx = 0.0;
  for (int m0 = 0; m0 < n; m0 += 256) {
    double v[4], x[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int m = m0 + 64 * q + lane;
      v[q] = m < n ? xload(p + m) : 0.0;
      x[q] = p2 && m < n ? xload(p2 + m) : 0.0;
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int m = m0 + 64 * q + lane;
      if (m >= n) continue;
      w[q] += xpoll(p + m, v[q], sc);
      xstore(p + m, xsent());
      if (p2) {
        const double y = xpoll(p2 + m, x[q], sc);
        mx = (mx < y) ? y : mx;
        xstore(p2 + m, xsent());
      }
    }
  }
  GatherSumMax r;
#pragma unroll
  for (int q = 0; q < 4; q++)
    if (64 * q < n) w[q] = wave_sum(w[q]);  // uniform; a sum over no entry is +0
  r.sum = (w[0] + w[1]) + (w[2] + w[3]);
  r.max = p2 ? wave_max(mx) : 0.0;
  return r;
}

__global__ void k_fill_sentinel(int64_t n, double* __restrict__ x) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) x[i] = __longlong_as_double((long long)XSENT);
}

}  // namespace
