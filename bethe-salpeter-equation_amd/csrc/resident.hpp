// Kernels whose workgroups wait for one another while they run (the bulge
// chase resident in LDS, the panel of the one-stage reduction).
//
// Messages.  A double travels as one 16-byte word whose two 8-byte halves
// each carry 4 bytes of it and a 4-byte tag, written by one device-coherent
// store and polled by device-coherent loads until both tags are the wanted
// ones: the data itself says when it is there, so nothing waits for a store to
// complete before a flag is written (8-byte accesses are single-copy atomic).
// Tags grow along a run and the buffers start zeroed, so a stale word never
// matches.  Measured: 0.44 us from a store to the polling reader inside an
// XCD, 0.6 us across XCDs.
//
// Residency.  Such a kernel needs all its workgroups on the device at once.
// They meet at a counter before they touch anything; when that does not
// happen within RS_MEET_TICKS they leave together and report 2, and the caller
// takes a path without this need.  Two such kernels at once could each hold
// part of the device and wait for the rest, so the launches of one process on
// a device follow one another (resident_launch: each waits, on the device, for
// the event of the one before).
#pragma once
#include "bse_common.hpp"
#include <functional>

#define RS_COHERENT 16                         // cache policy of a device-coherent buffer access (sc1)
#define RS_SPIN (1u << 23)                     // polls (each a memory round trip) before a wait is given up
#define RS_MEET_TICKS 200000000ull             // 2 s of the 100 MHz clock
#define RS_ABORT 0x80000000u

hipError_t resident_launch(int device, hipStream_t st, const std::function<hipError_t()>& launch);

__device__ inline bse_i4v rs_word(double v, int tag) {
    const bse_i4v w = {__double2loint(v), tag, __double2hiint(v), tag};
    return w;
}
__device__ inline bool rs_here(bse_i4v w, int tag) { return w[1] == tag && w[3] == tag; }
__device__ inline double rs_value(bse_i4v w) { return __hiloint2double(w[2], w[0]); }

// The host's refusal, for tests of what follows one: the counter starts with the
// abort bit, so every workgroup leaves from rs_meet.
inline hipError_t rs_refuse(hipStream_t st, unsigned* meet) {
    static const unsigned abort_bit = RS_ABORT;
    return hipMemcpyAsync(meet, &abort_bit, sizeof(abort_bit), hipMemcpyHostToDevice, st);
}

// All workgroups resident?  An arrival adds one; a workgroup that has waited
// too long sets RS_ABORT, and only while the count is short (compare and
// swap), so either every workgroup sees the full count or every one leaves.
__device__ inline bool rs_meet(unsigned* meet, unsigned all, int* err) {
    unsigned v = __hip_atomic_fetch_add(meet, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u;
    const unsigned long long t0 = wall_clock64();
    for (;;) {
        if (v & RS_ABORT) break;
        if (v == all) return true;
        if (wall_clock64() - t0 > RS_MEET_TICKS) {
            unsigned want = v;
            if (__hip_atomic_compare_exchange_strong(meet, &want, v | RS_ABORT, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT))
                break;
            v = want;
            continue;
        }
        __builtin_amdgcn_s_sleep(4);
        v = __hip_atomic_load(meet, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __hip_atomic_store(err, 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return false;
}

// One failed poll: true when the wait is to be given up.
__device__ inline bool rs_give_up(unsigned& spins, int* err) {
    ++spins;
    if ((spins & 1023u) == 0 && __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return true;
    if (spins > RS_SPIN) {
        __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return true;
    }
    return false;
}

