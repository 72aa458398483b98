// wave.h -- device helpers shared by the kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ct2 {

// Orders the wave's LDS accesses before and after it: what the lanes wrote is
// read by the others.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Adds v to the sum s, the rounding error to c.
__device__ __forceinline__ void two_sum(float& s, float& c, float v) {
#pragma clang fp contract(off)
    const float t = s + v;
    const float bp = t - s;
    const float e = (s - (t - bp)) + (v - bp);
    s = t;
    c += e;
}

// Counting-sort increment with one atomic per run of equal keys: every lane
// whose key is >= 0 adds 1 to counter[key] and receives the counter's value
// before its own increment (its slot in the key's segment).  Consecutive
// lanes with the same key form a run, and the run's first lane adds the run
// length in one atomic.  Inputs in spatial order (lattice or cell order) give
// long runs, so far fewer atomics meet at one counter.  Which slot a lane gets
// depends on the order the runs' atomics land in; the set of slots of a key is
// always 0 .. count-1.  Every lane of the wave must call it (inactive lanes with
// key < 0); the return value of an inactive lane is meaningless.
__device__ __forceinline__ int run_increment(int* counter, int key) {
    const int lane = (int)__lane_id();
    const int prev = __shfl_up(key, 1);
    const bool head = key >= 0 && (lane == 0 || prev != key);
    const uint64_t heads = __ballot(head);
    const uint64_t active = __ballot(key >= 0);
    const uint64_t upto = lane == 63 ? ~0ull : ((2ull << lane) - 1ull);  // lanes 0..lane
    // the run's first lane: the highest head at or below this lane
    const uint64_t below = heads & upto;
    const int start = below ? 63 - __clzll((long long)below) : lane;
    // the run ends at the next head or inactive lane above this one
    const uint64_t stop = (heads | ~active) & ~upto;
    const int end = stop ? __ffsll((long long)stop) - 1 : 64;
    int base = 0;
    if (head) base = atomicAdd(counter + key, end - lane);
    base = __shfl(base, start);
    return base + lane - start;
}

}  // namespace ct2
