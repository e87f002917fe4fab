// A small image in one launch: one workgroup runs the row tile, makes its
// stores visible to its own waves, then runs the column tile (the whole items
// of a batch).  For images whose rows and whose columns fit one 256-thread tile
// the second launch costs about what it saves on the device, and its enqueue on
// the host (device time, and time per call among others): 64 x 64 takes 5.5 and
// 6.3 us in one launch, 5.4 and 8.8 in two; 50 x 50 6.4 and 7.3, 6.7 and 8.9;
// 16 x 16 3.5 and 5.9, 3.8 and 8.9.  Which images take it: one_launch.  With 1024
// threads larger images fit, but one CU is then slower than two launches over
// many (100 x 37 13.2 us against 9.2, 61 x 67 18.4 against 9.9).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "batch_tile.hpp"

namespace mdft {

__global__ __launch_bounds__(WHOLE_THREADS) __attribute__((amdgpu_waves_per_eu(TILE_WAVES))) void k_whole(BatchJob row,
                                                                                                          BatchJob col)
{
    __shared__ float lds[batch_lds<WHOLE_THREADS, BATCH_ALL>()];
    // one copy of the tile code, two turns
    for (int turn = 0; turn < 2; ++turn) {
        const BatchJob bj = turn == 0 ? row : col;
        run_job<WHOLE_THREADS, BATCH_ALL>(bj, 0, lds);
        if (turn == 1) break;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __syncthreads();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    }
}

hipError_t launch_whole(const BatchJob& row, const BatchJob& col, hipStream_t stream)
{
    hipLaunchKernelGGL(k_whole, dim3(1), dim3(WHOLE_THREADS), 0, stream, row, col);
    return hipGetLastError();
}

// one word written, so the context loads this file's kernels at creation
__global__ void k_warm_whole(uint32_t* word)
{
    if (threadIdx.x == 0) word[0] = 0u;
}

hipError_t warm_whole(uint32_t* word, hipStream_t stream)
{
    hipLaunchKernelGGL(k_warm_whole, dim3(1), dim3(64), 0, stream, word);
    return hipGetLastError();
}

}  // namespace mdft
