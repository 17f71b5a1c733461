// Boundary-plane rings of the resident kernels (cvf_resident.hip, which
// describes the protocol; cvf_plane.hip): slots, tags and bounded waits.
#pragma once

#include "cvf_device.h"
#include "cvf_kernels.h"

namespace cvf {

// polls of one wait, of the order of a second: what the steps of a launch are
// delayed before they are done again by other launches
constexpr uint32_t kSpinLimit = 1u << 21;

// The version a slab publishes after the last step of a launch.
__device__ __forceinline__ uint64_t end_version(uint64_t step) { return step + 1; }

// Step-end planes: 64-bit ring words, the cell word in the low half and
// end_tag(step) in the high half, in ring slots kEndSlot, kEndSlot + 1 of
// the step's half.  The tag of a slot's previous contents (two steps back,
// or a stale value from before the rings were cleared) is never the tag a
// reader waits for.
constexpr uint32_t kEndSlot = kRingHalf - 2;
// first ring slot (of two) of the publish after half-sweep k
__device__ __forceinline__ uint32_t ring_slot(uint32_t k) { return 2 * k; }
__device__ __forceinline__ uint32_t end_tag(uint64_t step) { return launch_mark(step); }
__device__ __forceinline__ uint64_t ring_load64(const uint64_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void ring_store64(uint64_t* p, uint64_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Whether this launch, whose first step is step0, runs and keeps the lattice
// that it starts from: no launch before it was aborted.  `flag` is status[0],
// through the caches (as of the launch's start, or newer), loaded ahead of the
// lattice.
// The first workgroup of each XCD leaves the launch's mark, long before a wait
// of one that started after it can time out, so that workgroups which start
// after that know that the abort is theirs.  (One address for all: as an
// uncached load in every wavefront and a store in every workgroup these took
// 14 us of a launch of 512 workgroups.)
static __device__ __forceinline__ bool keeps_start(uint32_t flag, const uint32_t* status, uint64_t step0) {
  return !flag ||
         __hip_atomic_load(status + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == launch_mark(step0);
}
static __device__ __forceinline__ void leave_mark(const uint32_t* kept, uint32_t flag, uint32_t* status,
                                                  uint64_t step0) {
  if (kept && !flag && blockIdx.x < kNumXcd && threadIdx.x == 0)
    __hip_atomic_store(status + 1, launch_mark(step0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Wait until *v >= want.  False on time-out or abort.
static __device__ bool wait_version(const uint64_t* v, uint64_t want, uint32_t* status) {
  if (__hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return false;
  for (uint32_t it = 0;; ++it) {
    if (__hip_atomic_load(v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= want) {
      // no later load moves above the one that saw the version
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
      return true;
    }
    if ((it & 63u) == 63u && __hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return false;
    if (it >= kSpinLimit) {
      __hip_atomic_fetch_or(status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return false;
    }
    __builtin_amdgcn_s_sleep(2);
  }
}

// Load each of a lane's N words p[m] again until its tag (high half) is
// `tag`, starting from the values x[m] already loaded, in one loop of the
// whole wave: every pass checks all the words of every active lane, leaves
// when none is stale and reloads only the stale ones.  So every load is
// consumed on every path, and the compiler needs no wait for a load that
// might still be in flight later (on this GPU loads and stores share one
// counter, and such a wait would also wait out the ring stores).  False
// on time-out or abort (then some x[m] are stale).
template <int N>
__device__ __forceinline__ bool wait_tags(const uint64_t* const (&p)[N], uint32_t tag, uint64_t (&x)[N],
                                          uint32_t* status) {
  for (uint32_t it = 0;; ++it) {
    bool stale[N], any = false;
#pragma unroll
    for (int m = 0; m < N; ++m) {
      stale[m] = (uint32_t)(x[m] >> 32) != tag;
      any = any || stale[m];
    }
    if (!__ballot(any)) return true;
    if (((it & 63u) == 63u && __hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) ||
        it >= kSpinLimit) {
      __hip_atomic_fetch_or(status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return false;
    }
    __builtin_amdgcn_s_sleep(1);
#pragma unroll
    for (int m = 0; m < N; ++m)
      if (stale[m]) x[m] = ring_load64(p[m]);
  }
}

// Store a version after the workgroup barrier that follows the slot's ring
// stores (each writing wave waited for its stores to complete before it).
__device__ __forceinline__ void publish(uint64_t* v, uint64_t version) {
  __hip_atomic_store(v, version, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A writing wave's ring stores are complete (vmcnt 0) before it reaches the
// barrier after which the version is published.
__device__ __forceinline__ void ring_stores_done() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(0);
}

__device__ __forceinline__ uint32_t parity_of(int z, uint32_t L) { return (uint32_t)(z + (int)L) & 1u; }

// Cube c alone of the cube item eta_cube_item_q describes (random word
// rw = word c of the item's block): its eight corner words are half
// c ^ (the corner's swap) of the eight corner quads.
__device__ __forceinline__ void eta_cube_one_q(uint32_t* lds, uint32_t B, uint32_t U, const uint64_t* thr,
                                               const uint64_t* etab, uint32_t hL, uint32_t ox, uint32_t oy, uint32_t c,
                                               uint32_t rw) {
  const bool ex = ox + 1 == hL, ey = oy + 1 == hL;
  const uint32_t x1 = ex ? 0u : ox + 1, y1 = ey ? 0u : oy + 1;
  uint32_t idx[8], w[8];
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const uint32_t f = ((b & 1) && ex ? 2u : 0u) | ((b & 2) && ey ? 1u : 0u);
    idx[b] = ((b & 4) ? U : B) + 4 * (((b & 2) ? y1 : oy) * hL + ((b & 1) ? x1 : ox)) + (c ^ f);
  }
#pragma unroll
  for (int b = 0; b < 8; ++b) w[b] = lds[idx[b]];
  eta_cube_move(w, thr, etab, rw, [&](int b, uint32_t v) { lds[idx[b]] = v; });
}

}  // namespace cvf
