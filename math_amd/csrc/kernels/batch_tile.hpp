// Batched 2-D DFTs of mixed sizes.
//
// A batch is a list of work items over a table of axis jobs (one row job
// and one column job per image).  An item is one tile of one job, or a whole
// small image: a workgroup runs the row tile, makes its stores visible to its
// own waves, then runs the column tile, with no cross-workgroup
// synchronisation at all.  Three launch shapes share the item code:
//
//  * k_batch_grid: one workgroup per item, items laid out by the host so
//    each job runs on one XCD; a batch is two launches, whole images + row
//    tiles (256-thread tiles), then column tiles in the form that their number
//    calls for (column_kernel of the batch builder): 512 threads with two lines
//    per thread from 1024 points (16-4 columns for padded lengths 1024-4096, so
//    each row of a tile is a longer contiguous run, with two workgroups per CU),
//    512 with one, or 256.
//  * k_batch_persistent: a grid sized to the device's residency takes items
//    from a ticket counter, one launch per phase.
//  * k_batch_persistent with dependencies: one launch for everything; a
//    column tile waits on a per-image counter of finished row tiles (a
//    device-scope release/acquire pair per tile, which costs an L2
//    write-back per row tile).
//
// Every line runs the same per-line arithmetic as the single-image kernels
// (same radix schedule, explicit fmas), so a result is bitwise the same alone
// and in any mix.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fft_device.hpp"
#include "launch.hpp"
#include "smooth_device.hpp"

namespace mdft {

// The form of a shape a batch runs: two lines per thread where the shape has
// that in the kernels of two-line columns; one along rows, where two measured no
// better (4096^2: 140 us against 152), and for the columns of phase 1 (small
// whole images and single columns).
__host__ __device__ constexpr int batch_shape(int s, BatchHold hold)
{
    return has_x2(s) && hold == BATCH_COLS_X2 ? s | X2 : s;
}

template <int S, int T, BatchHold H>
constexpr int lds_need()
{
    if constexpr (tpl_of(S) > T) {
        return 0;
    } else {
        constexpr int a = H != BATCH_ALL ? 0 : LineCfg<batch_shape(S, H), T>::template lds_floats<false>();
        constexpr int b = LineCfg<batch_shape(S, H), T>::template lds_floats<true>();
        return a > b ? a : b;
    }
}

constexpr int cmax(int a, int b) { return a > b ? a : b; }

template <int T, BatchHold C>
constexpr int batch_lds()
{
    return cmax(gen_lds_floats(T),
           cmax(cmax(cmax(cmax(lds_need<5, T, C>(), lds_need<6, T, C>()), cmax(lds_need<7, T, C>(), lds_need<8, T, C>())),
                     cmax(cmax(cmax(lds_need<9, T, C>(), lds_need<10, T, C>()),
                               cmax(lds_need<11, T, C>(), lds_need<12, T, C>())),
                          lds_need<13, T, C>())),
                cmax(cmax(cmax(lds_need<F3_BASE + 6, T, C>(), lds_need<F3_BASE + 7, T, C>()),
                          cmax(lds_need<F3_BASE + 8, T, C>(), lds_need<F3_BASE + 9, T, C>())),
                     cmax(lds_need<F3_BASE + 10, T, C>(), lds_need<F3_BASE + 11, T, C>()))));
}

// One variant.  The thread and tile indices go through an empty asm of its own in every
// variant: otherwise the index arithmetic the variants share is hoisted above
// the dispatch and held there in registers that the variants then spill.
template <int S, int T, bool BLUE, bool COLS>
__device__ __forceinline__ void run_variant(const AxisJob& job, int tile, float* lds)
{
    int tid = threadIdx.x;
    asm volatile("; tile variant %2" : "+v"(tid), "+s"(tile) : "n"(S * 4 + (BLUE ? 2 : 0) + (COLS ? 1 : 0)));
    line_tile<S, T, BLUE, COLS>(job, tile, lds, tid);
}

template <int S, int T, BatchHold H, bool COLS>
__device__ __forceinline__ void run_axis(const AxisJob& job, int blue, int tile, float* lds)
{
    if constexpr (S >= 2) {
        if (blue) {
            run_variant<batch_shape(S, H), T, true, COLS>(job, tile, lds);
            return;
        }
    }
    run_variant<batch_shape(S, H), T, false, COLS>(job, tile, lds);
}

// a smooth length (its own asm for the indices, like run_variant)
template <int T, bool COLS>
__device__ __forceinline__ void run_smooth(const AxisJob& job, int tile, float* lds)
{
    int tid = threadIdx.x;
    asm volatile("; tile variant %2" : "+v"(tid), "+s"(tile) : "n"(GEN_SHAPE * 4 + (COLS ? 1 : 0)));
    smooth_tile<T, COLS>(job, tile, lds, tid);
}

template <int S, int T, BatchHold H>
__device__ __forceinline__ void run_tile_body(const AxisJob& job, int blue, int cols, int tile, float* lds)
{
    if constexpr (S == GEN_SHAPE) {
        if constexpr (H != BATCH_ALL)
            run_smooth<T, true>(job, tile, lds);
        else if (cols)
            run_smooth<T, true>(job, tile, lds);
        else
            run_smooth<T, false>(job, tile, lds);
    } else if constexpr (tpl_of(S) <= T) {
        if constexpr (H != BATCH_ALL)
            run_axis<S, T, H, true>(job, blue, tile, lds);
        else if (cols)
            run_axis<S, T, H, true>(job, blue, tile, lds);
        else
            run_axis<S, T, H, false>(job, blue, tile, lds);
    }
}

template <int S, int T>
__device__ __noinline__ void run_tile_call(const BatchJob* jobs, uint32_t job, int tile, float* lds);

// Grid kernels inline every variant (register allocation per region,
// occupancy-constrained); the persistent kernels call them out of line, since
// inlining into the ticket loop keeps too much alive across it.
template <int S, int T, bool INL, BatchHold H>
__device__ __forceinline__ void run_tile(const BatchJob* jobs, uint32_t job, const BatchJob& bj, int tile, float* lds)
{
    if constexpr (INL)
        run_tile_body<S, T, H>(bj.job, bj.blue, bj.cols, tile, lds);
    else
        run_tile_call<S, T>(jobs, job, tile, lds);
}

// Arguments of a call arrive in vector registers: the job is read again here,
// at a uniform address, so its fields are scalars in the tile code.
template <int S, int T>
__device__ __noinline__ void run_tile_call(const BatchJob* jobs, uint32_t job, int tile, float* lds)
{
    static_assert(sizeof(BatchJob) % 4 == 0, "copied by words");
    const uint64_t p = reinterpret_cast<uint64_t>(jobs + job);
    // the builtin returns a signed int: without the casts the low word's sign fills the high one
    const uint64_t u = (uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(p >> 32)))) << 32) |
                       uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(p)));
    auto words = reinterpret_cast<const __attribute__((address_space(4))) uint32_t*>(u);
    union Copy {
        uint32_t w[sizeof(BatchJob) / 4];
        BatchJob job;
        __device__ Copy() {}
    } copy;
#pragma unroll
    for (size_t i = 0; i < sizeof(BatchJob) / 4; ++i) copy.w[i] = words[i];
    const BatchJob& bj = copy.job;
    run_tile_body<S, T, BATCH_ALL>(bj.job, bj.blue, bj.cols, __builtin_amdgcn_readfirstlane(tile), lds);
}

// every shape a batch runs
#define MDFT_BATCH_SHAPES(X)                                                                           \
    X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(F3_BASE + 6) X(F3_BASE + 7) \
    X(F3_BASE + 8) X(F3_BASE + 9) X(F3_BASE + 10) X(F3_BASE + 11) X(GEN_SHAPE)

template <int T, bool INL, BatchHold H>
__device__ __forceinline__ void run_job_tile(const BatchJob* jobs, uint32_t job, int tile, float* lds)
{
    const BatchJob bj = jobs[job];
    switch (bj.shape) {
#define MDFT_CASE(S) \
    case S: run_tile<S, T, INL, H>(jobs, job, bj, tile, lds); break;
        MDFT_BATCH_SHAPES(MDFT_CASE)
#undef MDFT_CASE
    default: break;
    }
}

// the same for a job given by value (inlined)
template <int T, BatchHold H>
__device__ __forceinline__ void run_job(const BatchJob& bj, int tile, float* lds)
{
    switch (bj.shape) {
#define MDFT_CASE(S) \
    case S: run_tile_body<S, T, H>(bj.job, bj.blue, bj.cols, tile, lds); break;
        MDFT_BATCH_SHAPES(MDFT_CASE)
#undef MDFT_CASE
    default: break;
    }
}

// One item; every branch is on a wave-uniform value.
template <int T, bool INL, BatchHold H>
__device__ __forceinline__ void run_item(const BatchJob* __restrict__ jobs, uint2 item, float* lds)
{
    const uint32_t x = __builtin_amdgcn_readfirstlane(item.x);
    const uint32_t y = __builtin_amdgcn_readfirstlane(item.y);
    // one copy of the tile code: a whole image takes two turns (rows, columns)
    const bool whole = (y & BATCH_WHOLE) != 0;
    uint32_t job = x;
    int tile = whole ? 0 : (int)y;
    for (int turn = 0;; ++turn) {
        run_job_tile<T, INL, H>(jobs, job, tile, lds);
        if (!whole || turn == 1) break;
        // the column tile reads what this workgroup's waves just stored
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __syncthreads();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        job = y & ~BATCH_WHOLE;
    }
}

}  // namespace mdft
