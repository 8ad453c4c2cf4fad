// rotate.hpp -- wavefronts of one launch taking turns on the SIMDs.
//
// A grid of, say, 1.4 wavefronts per SIMD launched at once leaves most SIMDs
// one wavefront and some two, and ends when those two do.  A rotating launch
// starts a whole number of wavefronts per SIMD; each takes the next ticket of
// the run (chunk c of group g is ticket c * groups + g), loads the group's lane
// state, advances it over the chunk's ticks and parks it again.  The lane
// programs give the same bits however their ticks are cut.  rotate_plan.hpp
// says when this is used and what it measured.
#pragma once

#include <hip/hip_runtime.h>

#include "runtime.hpp"

namespace chaos {

// Device control block: the ticket counter, an error word and, per group, the
// chunks done.
struct RotateCtl {
    unsigned* head;
    int* err;
    unsigned* done;  // [groups]
    unsigned groups;
    unsigned chunks;
};

// A wave-uniform value kept in VGPRs (every lane a copy) while the code between
// put() and get() needs the SGPRs: the step maps' coefficients and the wave
// masks of the detector fill them, and what a rotating launch keeps across a
// group's ticks would be spilled lane by lane inside the hot loops instead
// (Chameleon peak map of 300^2 points: 33.6 ms without, 31.3 ms with it).
template <class T>
struct InVgprs {
    static_assert(sizeof(T) % 4 == 0, "whole registers");
    static constexpr int N = sizeof(T) / 4;
    unsigned w[N];
    __device__ __forceinline__ explicit InVgprs(const T& v)
    {
        __builtin_memcpy(w, &v, sizeof v);
#pragma unroll
        for (int k = 0; k < N; ++k) asm volatile("" : "+v"(w[k]));
    }
    __device__ __forceinline__ T get() const
    {
        unsigned u[N];
#pragma unroll
        for (int k = 0; k < N; ++k) u[k] = __builtin_amdgcn_readfirstlane(w[k]);
        T v;
        __builtin_memcpy(&v, u, sizeof v);
        return v;
    }
};

// Polls of a wait before it is given up (a poll takes 0.5 to 1 us; the chunk
// waited for takes 10 s at most, kRotateChunkSteps).
constexpr unsigned kRotatePolls = 1u << 27;

// body(group, chunk, lane) for every ticket.  A ticket's predecessor (the same
// group's chunk before it) was handed out earlier, to a wavefront that is
// running -- only running wavefronts take tickets -- and each holds one ticket
// at a time, so the wait for it ends; every wavefront leaves when the tickets
// are used up.  A wait that does not end all the same is given up after
// kRotatePolls: the error word is set, the wavefront leaves, and the host
// reports the call as failed.  The state crosses the XCDs' L2 caches between
// chunks: parked and released at agent scope, acquired before it is loaded.
//
// Lane 0 takes the ticket for the wave, so the lanes must come to it together.
// Every trip ends in a wave barrier: the compiler may not put it under a further
// condition, so lanes that skip a divergent tail of the body meet the others
// there before the back edge.  That is how it treats the barrier, not something
// the barrier promises, so each trip begins by looking at which lanes are
// active: a wavefront that is not whole sets the error word and leaves, and the
// call fails instead of taking a ticket with some of its lanes.  (An earlier
// form ended the loop in `if (lane == 0) store`; the other lanes took the back
// edge alone and read ticket 0 for ever.)
template <class Body>
__device__ __forceinline__ void rotate(const RotateCtl& args, Body&& body)
{
    const int lane = threadIdx.x & 63;
    const InVgprs<RotateCtl> kept(args);
    struct Ticket {
        unsigned g, c, trip;
    };
    unsigned trip = 0;
    for (;;) {
        const RotateCtl ctl = kept.get();
        if (__builtin_amdgcn_ballot_w64(true) != ~0ull) {
            __hip_atomic_store(ctl.err, 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            break;
        }
        const unsigned total = ctl.groups * ctl.chunks;
        // one ticket a wave: lane 0 takes it (the lanes are together here).  An
        // add by all 64 lanes would hand out 64 numbers, which are one atomic
        // only where the compiler happens to combine them
        unsigned t = 0;
        if (lane == 0)
            t = __hip_atomic_fetch_add(ctl.head, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_wave_barrier();
        t = __builtin_amdgcn_readfirstlane(t);
        if (t >= total || trip > total) break;
        const unsigned c = t / ctl.groups, g = t - c * ctl.groups;
        if (c > 0) {
            unsigned polls = 0;
            while (__builtin_amdgcn_readfirstlane(__hip_atomic_load(ctl.done + g, __ATOMIC_RELAXED,
                                                                    __HIP_MEMORY_SCOPE_AGENT)) < c &&
                   ++polls < kRotatePolls)
                __builtin_amdgcn_s_sleep(16);
            if (polls == kRotatePolls) {
                __hip_atomic_store(ctl.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
        const InVgprs<Ticket> ticket(Ticket{g, c, trip});
        body(g, c, lane);
        __builtin_amdgcn_wave_barrier();
        const Ticket mine = ticket.get();
        const RotateCtl after = kept.get();
        if (mine.c + 1 < after.chunks) {
            // every lane stores the same word: no divergent branch
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            __hip_atomic_store(after.done + mine.g, mine.c + 1, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
        trip = mine.trip + 1;
        __builtin_amdgcn_wave_barrier();
    }
}

// Control block in call scratch, cleared on the call's stream (a kernel, not a
// memset); its error word is checked at the end of the timed region
// (CallCtx::end).
RotateCtl make_rotate_ctl(CallCtx& ctx, long long groups, long long chunks);
// Blocks of `block` threads that put `waves` wavefronts on every SIMD.
unsigned rotate_grid(CallCtx& ctx, int waves, int block = 256);
// SIMDs of the call's device (four per CU).
long long device_simds(CallCtx& ctx);

}  // namespace chaos
