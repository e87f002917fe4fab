// The batch kernels of one workgroup size and content: compiled once each
// (MDFT_BATCH_T = 256, 512, 1024, MDFT_BATCH_HOLD = a BatchHold) and for 256 also
// as the persistent shapes (MDFT_BATCH_PERSISTENT_TU = 1), since each holds many
// tile variants.  Row tiles and whole images take 256 threads (a line of every
// batched length fits those), so the larger sizes hold column tiles only.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "batch_tile.hpp"

namespace mdft {

#if !MDFT_BATCH_PERSISTENT_TU

// Four waves per SIMD (<= 128 VGPRs): 256-thread tiles (4 workgroups per
// CU), 512-thread tiles (two) or 1024-thread tiles (one).
template <int T, BatchHold H>
__global__ __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(TILE_WAVES))) void k_batch_grid(
    const BatchJob* __restrict__ jobs, const uint2* __restrict__ items)
{
    __shared__ float lds[batch_lds<T, H>()];
    // the host lays items out per XCD (block b runs on XCD b % 8)
    run_item<T, true, H>(jobs, items[blockIdx.x], lds);
}

static_assert(batch_holds(MDFT_BATCH_T, BatchHold(MDFT_BATCH_HOLD)), "a size and content launch_batch_grid knows");

template <>
hipError_t launch_batch_grid_t<MDFT_BATCH_T, BatchHold(MDFT_BATCH_HOLD)>(const BatchJob* jobs, const uint2* items,
                                                                         uint32_t nitems, hipStream_t stream)
{
    hipLaunchKernelGGL((k_batch_grid<MDFT_BATCH_T, BatchHold(MDFT_BATCH_HOLD)>), dim3(nitems), dim3(MDFT_BATCH_T), 0,
                       stream, jobs, items);
    return hipGetLastError();
}

template <int T, BatchHold H>
__global__ void k_warm_batch_grid(uint32_t* word)
{
    if (threadIdx.x == 0) word[0] = 0u;
}

template <>
hipError_t warm_batch_grid<MDFT_BATCH_T, BatchHold(MDFT_BATCH_HOLD)>(uint32_t* word, hipStream_t stream)
{
    hipLaunchKernelGGL((k_warm_batch_grid<MDFT_BATCH_T, BatchHold(MDFT_BATCH_HOLD)>), dim3(1), dim3(64), 0, stream,
                       word);
    return hipGetLastError();
}

#else

// The item loop contains barriers, so its control flow is kept free of
// lane-divergent regions: every branch tests a value broadcast with
// readfirstlane or a wave index, and single-lane atomics are issued by the
// whole wave with an increment of 1 on lane 0 and 0 elsewhere.  (A
// thread-0-only region inside the loop lets the compiler rotate the loop so
// the other lanes reach the next barrier without passing the ticket update.)
// Deadlock freedom of the dependency mode: an item waits only on items with
// smaller tickets, taken by running workgroups that never wait on later ones.
template <int T>
__global__ __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(TILE_WAVES))) void k_batch_persistent(
    const BatchJob* __restrict__ jobs, const uint2* __restrict__ items, uint32_t nitems, uint32_t* ctl,
    uint32_t spin_limit)
{
    __shared__ float lds[batch_lds<T, BATCH_ALL>()];
    __shared__ uint32_t s_item;
    uint32_t* ticket = ctl;
    uint32_t* err = ctl + 1;
    uint32_t* counters = ctl + BATCH_CTL_HEADER;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x) >> 6;
    const uint32_t one_on_lane0 = (threadIdx.x & 63) == 0 ? 1u : 0u;
    for (;;) {
        if (wave == 0) {
            const uint32_t t = atomicAdd(ticket, one_on_lane0);
            s_item = __builtin_amdgcn_readfirstlane(t);
        }
        __syncthreads();
        const uint32_t it = __builtin_amdgcn_readfirstlane(s_item);
        __syncthreads();
        if (it >= nitems) break;
        const uint2 item = items[it];
        const BatchJob bj = jobs[__builtin_amdgcn_readfirstlane(item.x)];
        if (bj.dep >= 0) {
            // every wave polls the image's row counter itself, then acquires
            uint32_t spins = 0;
            for (;;) {
                const uint32_t c = __builtin_amdgcn_readfirstlane(
                    __hip_atomic_load(&counters[bj.dep], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                if (c >= (uint32_t)bj.dep_need) break;
                if (++spins > spin_limit) {
                    atomicOr(err, one_on_lane0);
                    break;
                }
                __builtin_amdgcn_s_sleep(2);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
        run_item<T, false, BATCH_ALL>(jobs, item, lds);
        if (bj.sig >= 0) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");  // release this wave's stores
            __syncthreads();
            if (wave == 0) atomicAdd(&counters[bj.sig], one_on_lane0);
        }
    }
}

template <>
hipError_t launch_batch_persistent_t<MDFT_BATCH_T>(const BatchJob* jobs, const uint2* items, uint32_t nitems,
                                                   uint32_t* ctl, int grid, uint32_t spin_limit, hipStream_t stream)
{
    hipLaunchKernelGGL(k_batch_persistent<MDFT_BATCH_T>, dim3(grid), dim3(MDFT_BATCH_T), 0, stream, jobs, items,
                       nitems, ctl, spin_limit);
    return hipGetLastError();
}

template <>
hipError_t batch_occupancy_t<MDFT_BATCH_T>(int* blocks_per_cu)
{
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, k_batch_persistent<MDFT_BATCH_T>, MDFT_BATCH_T,
                                                        0);
}

template <int T>
__global__ void k_warm_batch_persistent(uint32_t* word)
{
    if (threadIdx.x == 0) word[0] = 0u;
}

template <>
hipError_t warm_batch_persistent<MDFT_BATCH_T>(uint32_t* word, hipStream_t stream)
{
    hipLaunchKernelGGL(k_warm_batch_persistent<MDFT_BATCH_T>, dim3(1), dim3(64), 0, stream, word);
    return hipGetLastError();
}

#endif

}  // namespace mdft
