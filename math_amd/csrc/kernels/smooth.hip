// Axis passes over lines of smooth length (smooth_device.hpp): one image, the
// image path, and the tables of a length.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "launch.hpp"
#include "smooth_device.hpp"

namespace mdft {

template <int T, bool COLS>
__global__ __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(TILE_WAVES))) void k_smooth(AxisJob job)
{
    __shared__ float lds[gen_lds_floats(T)];
    smooth_tile<T, COLS>(job, COLS ? xcd_remap(blockIdx.x, gridDim.x) : blockIdx.x, lds, threadIdx.x);
}

template <int T, bool COLS, int IO>
__global__ __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(TILE_WAVES))) void k_smooth_image(AxisJob job,
                                                                                                     ImageIO io)
{
    __shared__ float lds[gen_lds_floats(T)];
    smooth_tile<T, COLS, IO>(job, COLS ? xcd_remap(blockIdx.x, gridDim.x) : blockIdx.x, lds, threadIdx.x, io);
}

// workgroups of a pass, 0 for none; the job's lines must fit the workgroup
static hipError_t smooth_grid(const AxisJob& job, int threads, unsigned* grid)
{
    *grid = 0;
    if (job.count < 0 || job.tpl < 1 || job.tpl > threads || job.n > 16 * job.tpl || job.npass < 2 ||
        job.npass > GEN_MAX_PASS)
        return hipErrorInvalidValue;
    const int64_t lines = threads / job.tpl;
    const int64_t g = (int64_t(job.count) + lines - 1) / lines;
    if (g > 0x7fffffff) return hipErrorInvalidValue;
    *grid = (unsigned)g;
    return hipSuccess;
}

template <int T>
static hipError_t launch_smooth_t(const AxisJob& job, bool cols, hipStream_t stream)
{
    unsigned grid;
    const hipError_t e = smooth_grid(job, T, &grid);
    if (e != hipSuccess || grid == 0) return e;
    if (cols)
        hipLaunchKernelGGL((k_smooth<T, true>), dim3(grid), dim3(T), 0, stream, job);
    else
        hipLaunchKernelGGL((k_smooth<T, false>), dim3(grid), dim3(T), 0, stream, job);
    return hipGetLastError();
}

hipError_t launch_smooth(const AxisJob& job, bool cols, int threads, hipStream_t stream)
{
    switch (threads) {
    case 64: return launch_smooth_t<64>(job, cols, stream);
    case 128: return launch_smooth_t<128>(job, cols, stream);
    case 256: return launch_smooth_t<256>(job, cols, stream);
    case 512: return launch_smooth_t<512>(job, cols, stream);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_smooth_image(const AxisJob& job, const ImageIO& io, bool cols, int mode, int threads,
                               hipStream_t stream)
{
    unsigned grid;
    const int T = cols && mode == IO_MAG && threads >= 512 ? 512 : 256;
    const hipError_t e = smooth_grid(job, T, &grid);
    if (e != hipSuccess || grid == 0) return e;
    const dim3 g(grid), b(T);
    if (!cols && mode == IO_LUM)
        hipLaunchKernelGGL((k_smooth_image<256, false, IO_LUM>), g, b, 0, stream, job, io);
    else if (!cols && mode == (IO_LUM | IO_MAG))
        hipLaunchKernelGGL((k_smooth_image<256, false, IO_LUM | IO_MAG>), g, b, 0, stream, job, io);
    else if (cols && mode == IO_MAG && T == 512)
        hipLaunchKernelGGL((k_smooth_image<512, true, IO_MAG>), g, b, 0, stream, job, io);
    else if (cols && mode == IO_MAG)
        hipLaunchKernelGGL((k_smooth_image<256, true, IO_MAG>), g, b, 0, stream, job, io);
    else if (cols && mode == (IO_LUM | IO_MAG))
        hipLaunchKernelGGL((k_smooth_image<256, true, IO_LUM | IO_MAG>), g, b, 0, stream, job, io);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

// the block of a length: the pass table, then the rows of every pass after the first
__global__ void k_gen_smooth(float2* out, GenPlan plan)
{
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx < GEN_MAX_PASS) {
        GenPass* table = reinterpret_cast<GenPass*>(out);
        table[idx] = plan.pass[idx];
    }
    int e = idx;
    for (int p = 1; p < plan.npass; ++p) {
        const int ns = plan.pass[p].ns, radix = plan.pass[p].radix;
        if (e < ns * 4) {
            const int64_t len = int64_t(ns) * radix;
            const int64_t q = (int64_t(e / 4) * tw_power(radix, e % 4)) % len;
            double s, c;
            sincospi(2.0 * (double)q / (double)len, &s, &c);
            out[GEN_TABLE + idx] = make_float2((float)c, (float)-s);
            return;
        }
        e -= ns * 4;
    }
}

int64_t smooth_block_len(const GenPlan& plan)
{
    int64_t len = GEN_TABLE;
    for (int p = 1; p < plan.npass; ++p) len += int64_t(plan.pass[p].ns) * 4;
    return len;
}

hipError_t gen_smooth(float2* out, const GenPlan& plan, hipStream_t stream)
{
    hipLaunchKernelGGL(k_gen_smooth, dim3((unsigned)((smooth_block_len(plan) + 255) / 256)), dim3(256), 0, stream, out,
                       plan);
    return hipGetLastError();
}

// one word written, so the context loads this file's kernels at creation
__global__ void k_warm_smooth(uint32_t* word)
{
    if (threadIdx.x == 0) word[0] = 0u;
}

hipError_t warm_smooth(uint32_t* word, hipStream_t stream)
{
    hipLaunchKernelGGL(k_warm_smooth, dim3(1), dim3(64), 0, stream, word);
    return hipGetLastError();
}

}  // namespace mdft
