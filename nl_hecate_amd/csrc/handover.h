// Work handed from workgroup to workgroup of one launch, in the order in which they started.
//
// What a workgroup does follows from the number that it draws when it starts, and it waits only for workgroups with lower
// numbers.  Those have started, and the lowest of them waits for nobody: so every wait ends, whatever part of the grid is resident
// and whatever else the device runs.
#pragma once
#include <hip/hip_runtime.h>

#include "runtime.h"

namespace nlh {

// A counter, in a cache line of its own, says how much of something is in memory.  The writer waits for its stores in every wave,
// meets its other waves at a barrier, and one wave makes them visible to the device and moves the counter (0.5 us).
constexpr int kTellStride = 32, kTellChunks = 4;   // a counter moves by that many chunks, and by single ones near the end
__device__ __forceinline__ void stores_arrived() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}
__device__ __forceinline__ void tell(unsigned *counter, int n) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __builtin_amdgcn_wave_barrier();
    if ((threadIdx.x & 63) == 0) __hip_atomic_store(counter, (unsigned)n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool told(const unsigned *counter, int until) {
    return __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= (unsigned)until;
}
// The whole workgroup, n counters of the first wave's lanes at once; what their writers stored before they told `until` is read
// behind this.
__device__ __forceinline__ void wait_told(const unsigned *counter, int n, int until) {
    if (threadIdx.x < 64) {
        const unsigned *mine = counter + ((int)threadIdx.x < n ? threadIdx.x : 0) * kTellStride;
        while (__builtin_amdgcn_ballot_w64(!told(mine, until))) __builtin_amdgcn_s_sleep(8);
    }
    __syncthreads();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
}

// The number that this workgroup draws from a counter; the same in every lane.  Tasks are drawn as
// well and not dealt out beforehand: a workgroup of the grid may find its place long after the others.
__device__ __forceinline__ int draw(unsigned *counter) {
    __shared__ int drawn;
    if (threadIdx.x == 0) drawn = (int)__hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const int n = __builtin_amdgcn_readfirstlane(drawn);
    __syncthreads();   // the next draw may follow at once
    return n;
}

constexpr int kAloneFloats = 81 * 256;   // more than half of a compute unit's LDS

__global__ static void clear_counters_kernel(unsigned *counters, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) counters[i] = 0;
}

// The counters of one launch, taken from a scratch slot and cleared; `at` is null where that is not free, or an error was raised.  They are held until the
// kernel is launched (they alone: other scratch of a call is for one host thread at a time), and cleared on the stream on which it has to be launched, `on`: with other host threads beside this one,
// nobody else's kernel comes between, and nlh_set_stream does not part the two.  They are cleared behind their last user's
// kernel, since a workgroup that waits for a count that is taken away never ends: on the null stream, which cannot be destroyed, by the
// stream's order, on another by an event as well (scratch_event; 5 us between calls back to back).
struct Counters {
    const std::lock_guard<std::mutex> held{counters_in_use};
    const hipStream_t on = stream();
    unsigned *at;
    hipEvent_t used = nullptr;
    Counters(int slot, size_t n) : at(reinterpret_cast<unsigned *>(scratch_if_free(slot, n * sizeof(unsigned), on))) {
        if (at && on && !(used = scratch_event(slot))) at = nullptr;
        if (!at) return;
        const ErrorScope es;
        if (used) check_hip(hipStreamWaitEvent(on, used, 0), "counters: hipStreamWaitEvent");
        hipLaunchKernelGGL(clear_counters_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, on, at, (int)n);
        check_launch("clear_counters_kernel");
        if (es.failed()) at = nullptr;
    }
    Counters(const Counters &) = delete;
    ~Counters() {
        if (used && at) check_hip(hipEventRecord(used, on), "counters: hipEventRecord");
    }
};

}  // namespace nlh
