// Workgroups that stay on the chip for a whole solve and exchange data
// between themselves without ending the kernel.
//
// A solver iteration of a small system is two to nine launches of 4-8 us each,
// of which the arithmetic is a fraction of a microsecond: the launches, the
// ramp of every kernel and the reload of the matrix cost the rest.  A resident
// kernel keeps one workgroup per block of rows for all iterations.  What a
// workgroup hands to the others (vector entries, partial sums) is written and
// read with relaxed agent-scope atomics, which bypass the caches that are not
// coherent between XCDs; the writer waits for its stores to complete
// (s_waitcnt vmcnt(0)) before it publishes the partial sum that says so.
// Nothing is fenced: an agent-scope fence writes back or invalidates whole
// caches.  Measured for one exchange among resident workgroups (32 / 64 / 128 /
// 256 of them): 1.5 / 1.9 / 2.6 / 4.2 us this way, 4 / 7 / 13 / 28 us with
// release and acquire fences.
//
// A reduction is also the barrier: each workgroup publishes its partial sum in
// its own slot and every workgroup polls all slots until none holds the empty
// mark, then adds them in the fixed order of the launched kernels (1.8 / 2.2 /
// 2.4 / 2.8 us for 5 / 64 / 128 / 256 workgroups, both block sums included; 4.0
// for 256 with the slots side by side; 3.5-3.6 through one reducing workgroup
// that hands the total on).  Slots are used in a ring of kResRing generations.
// Emptying: once generation g is complete everyone has published g and so has
// finished reading g - 1; the owner then empties its slot of g - 1, and that
// store completes before its publication of g + 2 (it waits at every second one
// at least), hence before anyone polls g + 3 (the same ring entry).
//
// Every wait is bounded.  Before the first iteration the workgroups wait until
// all of them have started (they might not fit beside other work on the GPU)
// or the time limit has passed; then they leave, having written scratch only
// (the empty marks over p, zeros over z, x's copy).  One that gives up later
// leaves the others to give up at the exchanges it is missing from, or, at the
// last one, to finish and store their rows of x.  Either way `abort` is set, and
// the caller puts x back (restore_x) and runs the launched kernels instead.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

#include "mps_device.hpp"
#include "mps_internal.hpp"

namespace mps {

constexpr int kResRing = 4;
constexpr int kResSlots = 512;  // partial sums of one generation (one per workgroup)
constexpr int kResPitch = 8;    // a slot per 64-byte line: polls of one slot do not hold up a store to another
constexpr unsigned long long kResEmpty = ~0ull;  // no partial sum: NaNs are published as one quiet pattern

constexpr int kResWords64 = 4;  // values of one slot at most (a line holds 8)
// Why a solve was abandoned: a wait ended at its limit (some workgroups may have gone
// on), or a workgroup refused the system before any of them started.
constexpr unsigned kResGivenUp = 1, kResRefused = 2;
struct ResidentCtl {
  unsigned started;
  unsigned abort;  // kResGivenUp, kResRefused
  ResidentDrill drill;
  unsigned pad[22];
  long long out[32];  // results of a solve (read by the host together with the head)
  unsigned long long slot[kResRing][kResSlots * kResPitch];
};

static_assert(offsetof(ResidentCtl, slot) == kResHead, "what the host reads");

// Limits of the waits, in ticks of the constant 100 MHz clock: for the start
// (5 ms: other work on the GPU may hold the compute units) and for one
// generation (2 s: only a lost workgroup gets there).
constexpr long long kResStartTicks = 500000;
constexpr long long kResWaitTicks = 200000000;
struct Patience {
  long long start, wait;
};

template <class T>
__device__ __forceinline__ T agent_load(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void agent_store(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The wavefront's stores have completed at their destination.
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

template <bool DRILL>
__device__ __forceinline__ Patience resident_patience(const ResidentCtl* c) {
  if constexpr (DRILL) return Patience{c->drill.start_ticks, c->drill.wait_ticks};
  return Patience{kResStartTicks, kResWaitTicks};
}
// Before the stores of generation g: the workgroup that a drill holds back.
template <bool DRILL>
__device__ __forceinline__ void resident_hold(const ResidentCtl* c, unsigned g, unsigned idx) {
  if constexpr (DRILL) {
    if (g != c->drill.hold_generation || idx != c->drill.hold_group) return;
    const long long t0 = wall_clock64(), t = c->drill.hold_ticks;
    while (wall_clock64() - t0 < t) {
    }
  }
}

// Block-uniform; every thread calls it.  True once all workgroups of the grid
// have started and none has refused (ok == false).
__device__ __forceinline__ bool resident_start(ResidentCtl* c, bool ok, const Patience& w) {
  __shared__ int s_go;
  if (threadIdx.x == 0) {
    if (!ok) {
      agent_store(&c->abort, kResRefused);
      stores_done();
    }
    __hip_atomic_fetch_add(&c->started, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const long long t0 = wall_clock64();
    int go = 1;
    while (agent_load(&c->started) < gridDim.x) {
      if (agent_load(&c->abort)) {
        go = 0;
        break;
      }
      if (wall_clock64() - t0 > w.start) {
        agent_store(&c->abort, kResGivenUp);
        go = 0;
        break;
      }
    }
    if (agent_load(&c->abort)) go = 0;
    s_go = go;
  }
  __syncthreads();
  return s_go != 0;
}

// One thread: the workgroup's values of generation g.  Every wavefront has waited
// for its stores of older generations (slots and vector entries emptied) before
// the workgroup's last __syncthreads.
template <class... V>
__device__ __forceinline__ void resident_put(ResidentCtl* c, unsigned g, unsigned idx, V... values) {
  const double v[] = {values...};
#pragma unroll
  for (unsigned k = 0; k < sizeof...(V); k++) {
    const double t = (v[k] != v[k]) ? __builtin_nan("") : v[k];  // never the empty mark
    agent_store(&c->slot[g % kResRing][idx * kResPitch + k], static_cast<unsigned long long>(__double_as_longlong(t)));
  }
}
// The same after this thread's own wavefront's stores.
template <class... V>
__device__ __forceinline__ void resident_publish(ResidentCtl* c, unsigned g, unsigned idx, V... values) {
  stores_done();
  resident_put(c, g, idx, values...);
}

// Value `word` of workgroup k's slot of generation g.
__device__ __forceinline__ const double* resident_slot(const ResidentCtl* c, unsigned g, unsigned k, int word) {
  return reinterpret_cast<const double*>(&c->slot[g % kResRing][k * kResPitch + word]);
}
// It once it is published; ok: false if the wait was given up.
__device__ __forceinline__ double resident_word(ResidentCtl* c, unsigned g, unsigned k, int word, bool& ok,
                                                const Patience& w) {
  const unsigned long long* s = &c->slot[g % kResRing][k * kResPitch + word];
  unsigned long long b = agent_load(s);
  if (b == kResEmpty) {
    const long long t0 = wall_clock64();
    do {
      b = agent_load(s);
      if (b == kResEmpty && (agent_load(&c->abort) || wall_clock64() - t0 > w.wait)) {
        agent_store(&c->abort, kResGivenUp);
        ok = false;
        break;
      }
    } while (b == kResEmpty);
  }
  return __longlong_as_double(static_cast<long long>(b));
}

// Values word and word + 1 of workgroup k's slot, polled together.
__device__ __forceinline__ void resident_words(ResidentCtl* c, unsigned g, unsigned k, int word, bool& ok, double& v0,
                                               double& v1, const Patience& w) {
  const unsigned long long* s = &c->slot[g % kResRing][k * kResPitch + word];
  unsigned long long a = agent_load(s), b = agent_load(s + 1);
  if (a == kResEmpty || b == kResEmpty) {
    const long long t0 = wall_clock64();
    do {
      a = agent_load(s);
      b = agent_load(s + 1);
      if ((a == kResEmpty || b == kResEmpty) &&
          (agent_load(&c->abort) || wall_clock64() - t0 > w.wait)) {
        agent_store(&c->abort, kResGivenUp);
        ok = false;
        break;
      }
    } while (a == kResEmpty || b == kResEmpty);
  }
  v0 = __longlong_as_double(static_cast<long long>(a));
  v1 = __longlong_as_double(static_cast<long long>(b));
}

// Vectors whose entries say themselves that they are there: two buffers taken in
// turn, an entry is empty (all ones, a NaN that is never stored) until its owner
// has written it, and a reader polls the entries it needs.  So neither does the
// owner wait for its stores before it publishes the partial sum that goes with
// them, nor the reader for everyone's partial sum before it loads (the CG's
// iteration in k_cg_resident: 0.2 us less with 3 workgroups, 1.1-1.5 with 24 to
// 250).  Emptying: the exchange after the readers have used generation g
// (they publish theirs after it) tells the owner that all of them have; it then
// empties its entries, and that completes before it publishes again, hence
// before anyone polls the buffer for generation g + 2.
__device__ __forceinline__ bool flag_empty(double v) {
  return static_cast<unsigned long long>(__double_as_longlong(v)) == kResEmpty;
}
__device__ __forceinline__ void flag_clear(double* p) {
  agent_store(reinterpret_cast<unsigned long long*>(p), kResEmpty);
}
__device__ __forceinline__ void flag_store(double* p, double v) { agent_store(p, v != v ? __builtin_nan("") : v); }
// Entries p[0 .. N) once they are there; ok: false if the wait was given up.
template <int N, class T>
__device__ __forceinline__ void flag_wait(ResidentCtl* c, const T* const (&p)[N], T (&v)[N], bool& ok, const Patience& w) {
  auto look = [&] {
    bool there = true;
#pragma unroll
    for (int k = 0; k < N; k++) v[k] = agent_load(p[k]);
#pragma unroll
    for (int k = 0; k < N; k++) there = there && !flag_empty(v[k]);
    return there;
  };
  if (look()) return;
  const long long t0 = wall_clock64();
  while (!look())
    if (agent_load(&c->abort) || wall_clock64() - t0 > w.wait) {
      agent_store(&c->abort, kResGivenUp);
      ok = false;
      return;
    }
}

// After the whole workgroup has seen generation g complete: its slot of
// generation g - 1 is emptied (the first `words` values).
__device__ __forceinline__ void resident_empty(ResidentCtl* c, unsigned g, unsigned idx, unsigned words = 1) {
  if (threadIdx.x < words)
    agent_store(&c->slot[(g + kResRing - 1) % kResRing][idx * kResPitch + threadIdx.x], kResEmpty);
}

// Clears the control block (and whatever `extra` words of a status) before a
// resident launch: one launch of kResSlots threads.
__device__ __forceinline__ void resident_clear(ResidentCtl* c, const ResidentDrill& drill) {
  if (threadIdx.x == 0) {
    c->started = 0;
    c->abort = 0;
    c->drill = drill;
  }
  for (int g = 0; g < kResRing; g++)
    for (int k = threadIdx.x; k < kResSlots; k += blockDim.x)
      for (int w = 0; w < kResWords64; w++) c->slot[g][k * kResPitch + w] = kResEmpty;
}

}  // namespace mps
