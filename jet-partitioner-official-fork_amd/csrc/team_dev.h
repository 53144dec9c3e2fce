// Teams of workgroups on one XCD (device side): start-up, barrier, loads that
// see the other workgroups' stores.
//
// A device-wide barrier costs 5 us and more, because the XCDs' L2s are made
// coherent by writing them back. The CUs of one XCD share its L2, so a team of
// workgroups of one XCD needs no cache maintenance at all: stores are written
// through to the L2 and waited for (s_waitcnt) before the barrier, and
// everything another workgroup may have changed is read with agent-scope
// loads, which pass by the CU's own cache. Measured: 0.6 us per barrier and
// exchange for 8 workgroups, 0.9 us for 32, against 4.4 and 8.8 us for a
// device-wide barrier; an L2 hit takes about 0.1 us where a load after a
// kernel boundary takes 0.5 us.
//
// A launch starts eight workgroups (one per XCD in dispatch order) for each
// one wanted; each reads the number of its XCD, and those elsewhere end
// whenever they run. The first member starts the team as soon as the members
// wanted are there: it waits for nothing on the other XCDs, so two teams never
// wait for each other's CUs. It stops waiting when every workgroup of the
// launch has arrived (no member is to come) or the bound is reached, and then
// starts with the members there are, or abandons the team when they are too
// few (the host then takes the multi-kernel path). Members that come after the
// decision end at once. Every later wait is for members of a team that runs,
// and bounded too. A team of one is launched as one workgroup, on any XCD.
#pragma once
#include <hip/hip_runtime.h>

#include "conn_table.h"
#include "jet_types.h"
#include "team.h"

namespace jet {

constexpr int32_t TEAM_SPINS = 1 << 24;  // seconds: the members are resident

__device__ inline int64_t ldr64(const int64_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline uint64_t ldr64(const uint64_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline int32_t xcd_id() {
    return (int32_t)(__builtin_amdgcn_s_getreg(20 | (3 << 11)) & 15);  // HW_REG_XCC_ID, bits 0-3
}

enum : int32_t { TEAM_OUT = 0, TEAM_GO = 1, TEAM_ABANDON = 2 };

__device__ inline int32_t ceil_div_dev(int32_t a, int32_t b) { return (a + b - 1) / b; }

// Registers the calling workgroup (its thread 0) and decides: `go` becomes 1
// for the members of a team that runs, with its size (`need` to `wanted`) and
// the member's number. Returns TEAM_ABANDON to the one workgroup that has to
// report that the team was given up. max_spins: polls of the first member
// before it decides with the members there are (0: never a team).
__device__ inline int32_t team_start(TeamCtl& C, int32_t xcd, int32_t wanted, int32_t need, int32_t max_spins,
                                     int32_t& go, int32_t& size, int32_t& me) {
    if (wanted == 1) {  // launched alone, on whichever XCD
        go = size = 1;
        me = 0;
        return TEAM_GO;
    }
    go = 0;
    const bool here = xcd_id() == xcd;
    int32_t m = wanted;
    if (here) m = __hip_atomic_fetch_add(&C.members, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // ordered after the registration: a wait for the returned value
    asm volatile("s_waitcnt vmcnt(0)" ::"v"(m) : "memory");
    __hip_atomic_fetch_add(&C.arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (!here || m >= wanted) return TEAM_OUT;
    int32_t st = 0, spins = 0;
    if (m == 0) {
        while (ld_rx(&C.members) < wanted && ld_rx(&C.arrived) < (int32_t)gridDim.x && ++spins <= max_spins) {
        }
        const int32_t there = min(ld_rx(&C.members), wanted);
        st = there >= need && max_spins > 0 ? there : -1;
        __hip_atomic_store(&C.state, st, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
        while ((st = ld_rx(&C.state)) == 0 && ++spins <= TEAM_SPINS) {
        }
    }
    if (st > m) {
        go = 1;
        size = st;
        me = m;
        return TEAM_GO;
    }
    return m == 0 ? TEAM_ABANDON : TEAM_OUT;
}

// Barrier of the team's workgroups; false when a wait ran out (never, unless
// an invariant is broken: all members are resident).
struct Team {
    TeamCtl* c;
    int32_t size, me;
    uint32_t target = 0;
    int32_t* ok;  // LDS
    __device__ bool sync() {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // stores and atomics have reached the L2
        __syncthreads();
        if (size == 1) return *ok != 0;
        if (threadIdx.x == 0) {
            target += (uint32_t)size;
            __hip_atomic_fetch_add(&c->bar, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            int32_t spins = 0;
            while ((int32_t)(__hip_atomic_load(&c->bar, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - target) < 0) {
                if (++spins > TEAM_SPINS) {
                    *ok = 0;
                    atomicOr(&c->fail, 1);
                    break;
                }
            }
        }
        __syncthreads();
        return *ok != 0;
    }
};

// The workgroup's x-th own vertex: chunks of `own` consecutive vertices go to
// the team's workgroups in turn.
__device__ inline int64_t own_vertex(int32_t x, int32_t own, int32_t team, int32_t me) {
    return ((int64_t)(x / own) * team + me) * own + x % own;
}

}  // namespace jet
