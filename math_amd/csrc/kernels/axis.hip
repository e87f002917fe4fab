// Axis-pass kernels: one launch transforms every line of one axis of one
// image (the reference records rows_to_buffer, FFT, mul_d, FFT,
// rows_from_buffer as five dispatches per axis, src/gpu/dft/dft.cpp:326-347;
// here they are one fused kernel per axis).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fft_device.hpp"
#include "launch.hpp"

namespace mdft {

template <int S, int T, bool BLUE, bool COLS>
__global__ __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(TILE_WAVES))) void k_axis(AxisJob job)
{
    constexpr int LF = LineCfg<S, T>::template lds_floats<COLS>();
    __shared__ float lds[LF > 0 ? LF : 1];
    const int tile = COLS ? xcd_remap(blockIdx.x, gridDim.x) : blockIdx.x;
    line_tile<S, T, BLUE, COLS>(job, tile, lds, threadIdx.x);
}

template <int S, int T, bool COLS>
static hipError_t launch_axis_tt(const AxisJob& job, bool blue, hipStream_t stream)
{
    constexpr int LPW = LineCfg<S, T>::LPW;
    // in 64 bits: count may be up to 2^31 - 1
    const int64_t grid64 = (int64_t(job.count) + LPW - 1) / LPW;
    if (job.count < 0 || grid64 > 0x7fffffff) return hipErrorInvalidValue;
    if (grid64 == 0) return hipSuccess;
    const unsigned grid = (unsigned)grid64;
    if (blue) {
        if constexpr (base_of(S) >= 2 && (!(S & X2) || x2_tile(S, T, true)))
            hipLaunchKernelGGL((k_axis<S, T, true, COLS>), dim3(grid), dim3(T), 0, stream, job);
        else
            return hipErrorInvalidValue;
    } else {
        hipLaunchKernelGGL((k_axis<S, T, false, COLS>), dim3(grid), dim3(T), 0, stream, job);
    }
    return hipGetLastError();
}

// threads: 1024 or 512 = wide tiles (launch.hpp), 256 = narrow, 128 / 64 = small
// tiles for passes with few lines (clamped up to one line per workgroup)
template <int S, bool COLS>
static hipError_t launch_axis_t(const AxisJob& job, bool blue, bool x2, int threads, hipStream_t stream)
{
    constexpr int TPL = tpl_of(S);
    if (x2) {
        if constexpr (COLS && has_x2(S)) {
            if (threads >= 1024) return launch_axis_tt<S | X2, 1024, COLS>(job, blue, stream);
            if (threads >= 512) return launch_axis_tt<S | X2, 512, COLS>(job, blue, stream);
            return launch_axis_tt<S | X2, 256, COLS>(job, blue, stream);
        } else {
            return hipErrorInvalidValue;
        }
    }
    if constexpr (!(COLS && has_x2(S))) {
        if (threads >= 512 && threads > narrow_threads(S))
            return launch_axis_tt<S, wide_threads(S, COLS), COLS>(job, blue, stream);
    }
    if constexpr (TPL <= 64) {
        if (threads <= 64) return launch_axis_tt<S, 64, COLS>(job, blue, stream);
    }
    if constexpr (TPL <= 128) {
        if (threads <= 128) return launch_axis_tt<S, 128, COLS>(job, blue, stream);
    }
    return launch_axis_tt<S, narrow_threads(S), COLS>(job, blue, stream);
}

// one word written, so the context loads this file's kernels at creation
__global__ void k_warm_axis(uint32_t* word)
{
    if (threadIdx.x == 0) word[0] = 0u;
}

hipError_t warm_axis(uint32_t* word, hipStream_t stream)
{
    hipLaunchKernelGGL(k_warm_axis, dim3(1), dim3(64), 0, stream, word);
    return hipGetLastError();
}

template <bool COLS>
static hipError_t launch_axis_dir(int shape, const AxisJob& job, bool blue, int threads, hipStream_t stream)
{
    const bool x2 = (shape & X2) != 0;
    switch (base_of(shape)) {
    case 1: return launch_axis_t<1, COLS>(job, blue, x2, threads, stream);
    case 2: return launch_axis_t<2, COLS>(job, blue, x2, threads, stream);
    case 3: return launch_axis_t<3, COLS>(job, blue, x2, threads, stream);
    case 4: return launch_axis_t<4, COLS>(job, blue, x2, threads, stream);
    case 5: return launch_axis_t<5, COLS>(job, blue, x2, threads, stream);
    case 6: return launch_axis_t<6, COLS>(job, blue, x2, threads, stream);
    case 7: return launch_axis_t<7, COLS>(job, blue, x2, threads, stream);
    case 8: return launch_axis_t<8, COLS>(job, blue, x2, threads, stream);
    case 9: return launch_axis_t<9, COLS>(job, blue, x2, threads, stream);
    case 10: return launch_axis_t<10, COLS>(job, blue, x2, threads, stream);
    case 11: return launch_axis_t<11, COLS>(job, blue, x2, threads, stream);
    case 12: return launch_axis_t<12, COLS>(job, blue, x2, threads, stream);
    case 13: return launch_axis_t<13, COLS>(job, blue, x2, threads, stream);
    case 14: return launch_axis_t<14, COLS>(job, blue, x2, threads, stream);
    case F3_BASE + 6: return launch_axis_t<F3_BASE + 6, COLS>(job, blue, x2, threads, stream);
    case F3_BASE + 7: return launch_axis_t<F3_BASE + 7, COLS>(job, blue, x2, threads, stream);
    case F3_BASE + 8: return launch_axis_t<F3_BASE + 8, COLS>(job, blue, x2, threads, stream);
    case F3_BASE + 9: return launch_axis_t<F3_BASE + 9, COLS>(job, blue, x2, threads, stream);
    case F3_BASE + 10: return launch_axis_t<F3_BASE + 10, COLS>(job, blue, x2, threads, stream);
    case F3_BASE + 11: return launch_axis_t<F3_BASE + 11, COLS>(job, blue, x2, threads, stream);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_axis(int shape, const AxisJob& job, bool blue, bool cols, int threads, hipStream_t stream)
{
    return cols ? launch_axis_dir<true>(shape, job, blue, threads, stream)
                : launch_axis_dir<false>(shape, job, blue, threads, stream);
}

}  // namespace mdft
