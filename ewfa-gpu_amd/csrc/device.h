// device.h -- device helpers shared by the kernels' translation units.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ewfa {

// x with lane `lane` set to the uniform value v (v_writelane, whatever the
// exec mask).  The lane select goes through M0: one instruction reads one
// scalar register besides M0.
__device__ __forceinline__ int writelane_i32(int x, int v, int lane) {
    asm("v_writelane_b32 %0, %1, m0" : "+v"(x) : "s"(v), "{m0}"(lane));
    return x;
}

// Adds n to a work counter and returns its old value; with an `end`, a counter
// that has passed it is only read (one thread's call).
constexpr uint32_t NO_LOOK = 0xFFFFFFFFu;
__device__ __forceinline__ uint32_t counter_take(uint32_t* counter, uint32_t n, uint32_t end) {
    if (end != NO_LOOK) {
        const uint32_t now = __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (now >= end) return now;
    }
    return atomicAdd(counter, n);
}

// A wave's next work item from a counter: lane 0 adds n, every lane gets the
// old value.  The wave barrier joins the lanes' paths first: without it the
// compiler may thread a branch on the lane elsewhere in the caller's loop
// (`if (lane == 0) store`) past the add, into a loop of lanes 1..63 alone
// that reads the counter's value from a lane that never adds.
__device__ __forceinline__ uint32_t wave_take(uint32_t* counter, uint32_t n, int lane, uint32_t end = NO_LOOK) {
    __builtin_amdgcn_wave_barrier();
    uint32_t b = 0;
    if (lane == 0) b = counter_take(counter, n, end);
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)b);
}

// Synchronisation of the threads working on one pair.
template <int G>
__device__ __forceinline__ void group_sync() {
    if constexpr (G == 1) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
        __syncthreads();
    }
}

// Inclusive prefix sum over the 64 lanes with DPP only: row shifts by 1, 2,
// 4 and 8 within each row of 16 lanes, then lane 15 and lane 31 broadcast
// into the rows above.  Every lane of the wave must take part.
__device__ __forceinline__ int wave_incl_scan_i32(int x) {
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false);  // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false);  // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false);  // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false);  // row_shr:8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);  // row_bcast:15 into rows 1, 3
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false);  // row_bcast:31 into rows 2, 3
    return x;
}

// ---- CIGAR streams written by a wave -----------------------------------------

// Stream bytes of a match run of r bases: floor(r/127) bytes of -127, then
// -(r%127) when nonzero (src/kernels.cu:436-446).
__device__ __forceinline__ int run_bytes(int r) { return (r + 126) / 127; }

// A pair's stream region and the bytes of the stream so far (uniform).
struct WaveStream {
    int8_t* out;
    uint32_t cap, len;

    // a run at `at`, bytes at or past the region's end dropped
    __device__ __forceinline__ uint32_t put_run(uint32_t at, int r) const {
        for (; r >= 127; r -= 127, ++at)
            if (at < cap) out[at] = (int8_t)-127;
        if (r) {
            if (at < cap) out[at] = (int8_t)-r;
            ++at;
        }
        return at;
    }
    // lane by lane, a run and the op (OP_*) after it; lanes with act false add
    // nothing
    __device__ __forceinline__ void put(bool act, int run, int op) {
        const int nb = act ? run_bytes(run) + 1 : 0;
        const int incl = wave_incl_scan_i32(nb);
        if (act) {
            const uint32_t at = put_run(len + (uint32_t)(incl - nb), run);
            if (at < cap) out[at] = (int8_t)(op == 3 ? 'D' : op == 2 ? 'X' : 'I');
        }
        len += (uint32_t)__builtin_amdgcn_readlane(incl, 63);
    }
    // the last run and the terminator (zeros to the end of its dword, inside
    // the region), by one lane
    __device__ __forceinline__ void finish(int run, int lane) {
        const uint32_t end = len + (uint32_t)run_bytes(run);
        if (lane == 0) {
            put_run(len, run);
            const uint32_t stop = min((end & ~3u) + 4u, cap);
            for (uint32_t i = end; i < stop; ++i) out[i] = 0;
        }
        len = end;
    }
};

}  // namespace ewfa
