// batch_persist.hip -- the persistent launch of a batch.
#include "batch_blocks.hpp"

namespace mmx {

// ---------------------------------------------------- the persistent launch
//
// One cooperative launch (every workgroup resident) runs up to `tries` tries
// of the whole batch: the ten passes of a try and the controller one after
// another, separated by grid-wide barriers, each pass's virtual blocks dealt
// round-robin to the workgroups.  It stops early once no simulation is
// active.  A barrier wait is bounded: past kSpinLimit polls the workgroup
// records the time-out in `fail` and leaves; a timed-out barrier leaves the
// barrier words inconsistent, so the host resets them before the next launch.

constexpr long kSpinLimit = 1L << 25;

// Grid-wide barrier with agent-scope release/acquire (the workgroups of the
// 8 XCDs do not share an L2).  Returns false when the wait timed out.
__device__ bool grid_barrier(const PersistArgs &a)
{
    __shared__ int ok;
    __threadfence();
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned int gen =
            __hip_atomic_load(&a.bar[1], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned int arrived =
            __hip_atomic_fetch_add(&a.bar[0], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        ok = 1;
        if (arrived == gridDim.x - 1) {
            __hip_atomic_store(&a.bar[0], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_fetch_add(&a.bar[1], 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
        } else {
            long n = 0;
            while (__hip_atomic_load(&a.bar[1], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) ==
                   gen) {
                __builtin_amdgcn_s_sleep(2);
                if (++n > kSpinLimit) {
                    __hip_atomic_store(a.fail, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    ok = 0;
                    break;
                }
            }
        }
    }
    __syncthreads();
    __threadfence();
    return ok != 0;
}

template <int STAGE>
__device__ bool persist_passes(const BatchSim *__restrict__ sims, BatchState *__restrict__ st,
                               const PersistArgs &a, float2 *sm)
{
#define MMX_PASS(P, BODY)                                                                    \
    if (a.nblk[P] > 0) {                                                                     \
        for (int vb = blockIdx.x; vb < a.nblk[P]; vb += gridDim.x) {                         \
            BODY;                                                                            \
            __syncthreads(); /* the next tile reuses the LDS */                              \
        }                                                                                    \
        if (!grid_barrier(a)) return false;                                                  \
    }
    MMX_PASS(BP_XF, (bxf_block<STAGE, KIND_ANY>(sims, st, a.map[BP_XF], vb, sm)))
    MMX_PASS(BP_Y, (by_block<KIND_ANY>(STAGE, sims, st, a.map[BP_Y], vb, sm)))
    MMX_PASS(BP_Z, bz_block<KIND_ANY>(STAGE, sims, st, a.map[BP_Z], vb, sm))
    MMX_PASS(BP_YI, byi_block<KIND_ANY>(STAGE, sims, st, a.map[BP_YI], vb, sm))
    MMX_PASS(BP_XI, (bxi_block<STAGE, KIND_ANY>(sims, st, a.map[BP_XI], vb, sm)))
#undef MMX_PASS
    return true;
}

__global__ void __launch_bounds__(kBlock)
bpersist_kernel(const BatchSim *__restrict__ sims, BatchState *__restrict__ st, PersistArgs a)
{
    extern __shared__ float2 sm[];
    for (int k = 0; k < a.tries; k++) {
        if (!persist_passes<0>(sims, st, a, sm)) return;
        if (!persist_passes<1>(sims, st, a, sm)) return;
        if (blockIdx.x == 0) {
            for (int s = threadIdx.x; s < a.nsim; s += blockDim.x) control_one(st[s]);
            __syncthreads();
            if (threadIdx.x == 0) {
                int n = 0;
                for (int s = 0; s < a.nsim; s++) n += st[s].active;
                __hip_atomic_store(a.nactive, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        if (!grid_barrier(a)) return;
        if (__hip_atomic_load(a.nactive, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) return;
    }
}

const void *persist_kernel() { return reinterpret_cast<const void *>(bpersist_kernel); }

} // namespace mmx
