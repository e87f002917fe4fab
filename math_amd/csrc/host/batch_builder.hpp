// Construction of a batch's job table and work list, shared by the batch
// API and the server.
#pragma once

#include <cstdint>
#include <memory>
#include <vector>

#include "runtime.hpp"

namespace mdft {

struct BatchBuild {
    int threads_cols = BATCH_THREADS;  // workgroup size of column tiles
    BatchHold hold_cols = BATCH_ALL;  // and the kernel that runs them
    std::vector<BatchJob> jobs;
    std::vector<uint2> items;
    uint32_t nphase1 = 0;
    uint32_t ncounters = 0;
    std::vector<std::shared_ptr<const LinePlan>> keep;
};

// One transform of a batch: device pointers may be null and patched later
// through src_job/dst_job offsets (batch API) or given directly (server).
struct BatchEntry {
    uint32_t width, height;
    bool inverse;
    const float2* src;
    float2* dst;
};

// The tiles of one job: items (job, first), (job, first + 1), ..
struct TileGroup {
    int phase;
    int m, shape, blue, kind;  // kind: 0 a whole image, 1 row tiles, 2 column tiles
    uint32_t job, first, count;
    int64_t cost;  // of a tile: ~ points x passes (x2 for Bluestein's two FFTs, x2 for a whole image)
};
// Sorts groups by phase and kernel variant and writes the items of both phases
// (two words each) as their launches take them; returns the items of phase 1.
uint32_t lay_out_tiles(std::vector<TileGroup>& groups, uint32_t* words);

// Throws MDFT_ERR_SIZE where a side or its padded length is beyond the batch limit (8192).
void check_batch_sizes(const uint32_t* widths, const uint32_t* heights, size_t count);

// Builds jobs and items.  dependent: one-launch ordering with per-image
// counters; otherwise two phases sorted by kernel variant.  job_image[i]
// receives the index of the entry each job belongs to and job_is_col[i]
// whether it is the column job.
// threads_cols: column tiles, 512 for what column_kernel picks.
void build_batch(Context& ctx, const BatchEntry* entries, size_t count, int threads_cols, bool dependent,
                 BatchBuild& out, std::vector<uint32_t>* job_image = nullptr,
                 std::vector<uint8_t>* job_is_col = nullptr);

}  // namespace mdft
