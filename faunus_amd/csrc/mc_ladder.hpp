// Temperature ladders on the device: one round of swaps of a ladder's rungs, and the barrier
// at which the replicas of free-running ladders meet after each interval.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "mc_batch.hpp"
#include "philox.hpp"

namespace fmc {
namespace {

// One round of neighbour exchanges in one ladder (ParallelTempering, move.cpp:844-965):
// rungs k, k+1 for k of the round's parity, accepted with min(1, exp((b_a - b_b)(E_a -
// E_b))) on a Philox deviate of (round, ladder, k); an accepted swap exchanges the betas
// and the rung slots.
__device__ void swap_ladder_rungs(ReplicaState* states, int b, int m, int* rung_slot, int l, unsigned long long seed,
                                  unsigned long long round, unsigned long long* counters) {
    for (int k = static_cast<int>(round & 1); k + 1 < m; k += 2) {
        const int sa = rung_slot[b + k], sb = rung_slot[b + k + 1];
        ReplicaState& A = states[sa];
        ReplicaState& B = states[sb];
        const double x = (A.beta - B.beta) * (A.energy - B.energy);
        const Philox4 r = philox4x32_10(static_cast<uint32_t>(round), static_cast<uint32_t>(round >> 32),
                                        static_cast<uint32_t>(l), 0x5a5a0000u + static_cast<uint32_t>(k),
                                        static_cast<uint32_t>(seed), static_cast<uint32_t>(seed >> 32));
        const double u = (static_cast<double>(r.v[0] >> 5) * 67108864.0 + static_cast<double>(r.v[1] >> 6)) *
                         1.1102230246251565e-16;
        atomicAdd(&counters[0], 1ull);
        if (x >= 0.0 || u < exp(x)) {
            const double tb = A.beta;
            A.beta = B.beta;
            B.beta = tb;
            rung_slot[b + k] = sb;
            rung_slot[b + k + 1] = sa;
            atomicAdd(&counters[1], 1ull);
        }
    }
}

// The barrier of replica `rep`'s (S's) ladder after interval iv, by one thread, its energy written before:
// the energy is published before the arrival; the last replica to arrive swaps the rungs, the
// others wait for its release.  `beta` receives the replica's temperature label afterwards.
__device__ void ladder_barrier(const LadderRun& lr, int rep, ReplicaState* states, ReplicaState& S, int iv, double& beta) {
    const int l = lr.ladder_of[rep];
    if (l < 0) return;
    __threadfence();
    const unsigned target = static_cast<unsigned>(lr.size[l]) * static_cast<unsigned>(iv + 1);
    if (atomicAdd(&lr.arrive[l], 1u) + 1u == target) {
        __threadfence();
        swap_ladder_rungs(states, lr.begin[l], lr.size[l], lr.rung_slot, l, lr.seed,
                          lr.round0 + static_cast<unsigned long long>(iv), lr.counters);
        __threadfence();
        __hip_atomic_store(&lr.gen[l], static_cast<unsigned>(iv + 1), __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    } else {
        long long spins = 0;
        while (__hip_atomic_load(&lr.gen[l], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < static_cast<unsigned>(iv + 1)) {
            if (++spins > lr.spin_limit) {
                atomicMax(&S.error, 2); // a rung did not arrive: this replica stops
                break;
            }
            __builtin_amdgcn_s_sleep(20);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    beta = __hip_atomic_load(&S.beta, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

} // namespace
} // namespace fmc
