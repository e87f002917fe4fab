// Host side of the batch kernels: the launch by workgroup size (the kernels
// themselves are in batch_kernels.hip, one object per size and launch shape).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "batch_tile.hpp"

namespace mdft {

// longest padded length of a batch: one line of 8192 points takes 256 threads
constexpr int BATCH_MAXLOGM = 13;
static_assert(tpl_of(BATCH_MAXLOGM) <= BATCH_THREADS && tpl_of(F3_BASE + F3_MAX_K) <= BATCH_THREADS,
              "a line of every batched length fits a row tile");

__global__ void k_fill_u32(uint32_t* p, uint32_t n, uint32_t value)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = value;
}

hipError_t launch_batch_grid(int threads, BatchHold hold, const BatchJob* jobs, const uint2* items, uint32_t nitems,
                             hipStream_t stream)
{
    if (nitems == 0) return hipSuccess;
    if (!batch_holds(threads, hold)) return hipErrorInvalidValue;
    if (hold == BATCH_ALL) return launch_batch_grid_t<BATCH_THREADS, BATCH_ALL>(jobs, items, nitems, stream);
    if (hold == BATCH_COLS) return launch_batch_grid_t<512, BATCH_COLS>(jobs, items, nitems, stream);
    if (threads == 512) return launch_batch_grid_t<512, BATCH_COLS_X2>(jobs, items, nitems, stream);
    return launch_batch_grid_t<1024, BATCH_COLS_X2>(jobs, items, nitems, stream);
}

hipError_t warm_batch(uint32_t* word, hipStream_t stream)
{
    hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, stream, word, 1u, 0u);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = warm_batch_grid<BATCH_THREADS, BATCH_ALL>(word, stream);
    if (e == hipSuccess) e = warm_batch_grid<512, BATCH_COLS>(word, stream);
    if (e == hipSuccess) e = warm_batch_grid<512, BATCH_COLS_X2>(word, stream);
    if (e == hipSuccess) e = warm_batch_grid<1024, BATCH_COLS_X2>(word, stream);
    if (e == hipSuccess) e = warm_batch_persistent<BATCH_THREADS>(word, stream);
    return e;
}

hipError_t launch_batch_persistent(const BatchJob* jobs, const uint2* items, uint32_t nitems, uint32_t* ctl,
                                   uint32_t nctl, int grid, uint32_t spin_limit, hipStream_t stream)
{
    if (nitems == 0) return hipSuccess;
    // clear ticket, error flag and counters with a kernel (graph-capture safe)
    hipLaunchKernelGGL(k_fill_u32, dim3((nctl + 255) / 256), dim3(256), 0, stream, ctl, nctl, 0u);
    return launch_batch_persistent_t<BATCH_THREADS>(jobs, items, nitems, ctl, grid, spin_limit, stream);
}

int batch_lines_per_tile(int threads, BatchHold hold, int shape)
{
    if (shape < 1 || (!is_f3(shape) && shape > BATCH_MAXLOGM) ||
        (is_f3(shape) && (f3_k(shape) < F3_MIN_K || f3_k(shape) > F3_MAX_K)))
        return 0;
    const int tpl = tpl_of(shape);
    return tpl <= threads ? threads / tpl * lines_per_thread(batch_shape(shape, hold)) : 0;
}

hipError_t batch_occupancy(int* blocks_per_cu) { return batch_occupancy_t<BATCH_THREADS>(blocks_per_cu); }

int batch_max_logm() { return BATCH_MAXLOGM; }

}  // namespace mdft
