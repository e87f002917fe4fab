// Job tables and work lists of batched transforms.
//
// Each image contributes a row job and a column job, cut into tiles of whole
// lines.  A small image whose rows and columns each fit one tile becomes a
// single "whole" item done by one workgroup.  Without dependencies, the jobs'
// tile groups are sorted by phase (whole images and row tiles first, column tiles
// second) and then by kernel variant (padded length, Bluestein or not, axis)
// so neighbouring workgroups run the same code.  A line length gets the same
// radix schedule in every batch, so a result is bitwise the same alone or in
// any mix.
#include "batch_builder.hpp"

#include <algorithm>
#include <cmath>
#include <numeric>
#include <string>
#include <tuple>

#include "../../../include/mdft.h"

namespace mdft {

void check_batch_sizes(const uint32_t* widths, const uint32_t* heights, size_t count)
{
    const int limit = batch_max_logm();
    for (size_t i = 0; i < count; ++i) {
        compute_m(widths[i]);  // validates the sides
        compute_m(heights[i]);
        // the FFT lengths the tiles run (the padded length, or 3 * 2^k; a smooth length itself)
        for (int shape : {line_shape(widths[i], false), line_shape(heights[i], true)})
            if (shape != GEN_SHAPE && m_of(shape) > (1 << limit))
                throw Error(MDFT_ERR_SIZE, "batch transform " + std::to_string(i) + " (" + std::to_string(widths[i]) +
                                               "x" + std::to_string(heights[i]) +
                                               ") exceeds the batch padded-length limit " +
                                               std::to_string(1 << limit));
    }
}

// lines a tile holds of a plan's length
static int lines_per_tile(int threads, BatchHold hold, const LinePlan& lp)
{
    return lp.gen ? threads / lp.smooth.tpl : batch_lines_per_tile(threads, hold, lp.shape);
}
static int lines_per_tile(const LinePlan& lp) { return lines_per_tile(BATCH_THREADS, BATCH_ALL, lp); }

// whole images run both passes in one row-phase workgroup
static bool runs_whole(int w, int h, const LinePlan& row, const LinePlan& col)
{
    return w > 1 && h > 1 && h <= lines_per_tile(row) && w <= lines_per_tile(col);
}

// the tiles of a group in order
static uint32_t* write_tiles(const TileGroup& g, uint32_t* words)
{
    for (uint32_t t = 0; t < g.count; ++t) {
        *words++ = g.job;
        *words++ = g.first + t;
    }
    return words;
}

// cost of one line ~ points x passes
static double line_cost(const LinePlan& lp) { return double(lp.m) * (std::log2(double(lp.m)) + 2); }

// The kernel of the column phase: its tiles in the smallest form that still
// fills the device, since a tile's chain of loads, passes and exchanges takes as
// long as it has lines (us of the phase, 256 CUs):
//  * 256 threads while those tiles cost no more than one of the dearest per CU
//    (direct ones counted twice: they wait for memory, where the shorter runs
//    cost): 128 x 509 7.8 (10.0 in 512 threads with one line per thread, 14.4 with
//    two), 57 x 4093 20.3 (24.8, 25.4), 256 x 2238 15.6 (17.4, 18.2), but 256 x
//    4096 13.4 (10.8, 12.0);
//  * 512 threads and one line per thread below 1.5 tiles per CU of the two-line
//    form: 1024 x 1201 18.1 (18.3 with two), 2560 x 1021 22.3 (26.4); with two
//    above: 2048 x 1201 27.1 (30.5 with one), 2048 x 2047 30.6 (34.4); direct lines
//    gain more, tiles of 1536 and 3072 points count twice and of 4096 three times:
//    2048 x 1536 13.0 (14.5 with one), 1024 x 3072 16.5 (21.5), 512 x 4096 15.0 (15.6);
//  * one line per thread as well where no line has the two-line form (2048 x 4093
//    65.6, 70.4 in the kernel with two).
static BatchHold column_kernel(int TC, int cu_count, const BatchEntry* entries, size_t count,
                               const std::vector<std::shared_ptr<const LinePlan>>& plans)
{
    if (TC <= BATCH_THREADS) return BATCH_ALL;
    if (TC != BATCH_COL_THREADS) return BATCH_COLS_X2;
    double narrow = 0, dearest = 0;
    int64_t two = 0;
    bool any_two = false;
    for (size_t i = 0; i < count; ++i) {
        const int w = (int)entries[i].width, h = (int)entries[i].height;
        const LinePlan &row = *plans[2 * i], &col = *plans[2 * i + 1];
        if (w <= 1 || h <= 1 || runs_whole(w, h, row, col)) continue;
        const int n1 = lines_per_tile(col), n2 = lines_per_tile(TC, BATCH_COLS_X2, col);
        const double cost = n1 * line_cost(col);
        narrow += (w + n1 - 1) / n1 * cost * (col.blue ? 1 : 2);
        dearest = std::max(dearest, cost);
        const bool x2 = has_x2(col.shape);
        two += int64_t((w + n2 - 1) / n2) * (!x2 || col.blue ? 1 : col.m == 4096 ? 3 : is_f3(col.shape) ? 2 : 1);
        any_two |= x2;
    }
    if (narrow <= dearest * cu_count) return BATCH_ALL;
    return any_two && 2 * two >= 3 * int64_t(cu_count) ? BATCH_COLS_X2 : BATCH_COLS;
}

void build_batch(Context& ctx, const BatchEntry* entries, size_t count, int TC, bool dependent, BatchBuild& out,
                 std::vector<uint32_t>* job_image, std::vector<uint8_t>* job_is_col)
{
    out = BatchBuild{};
    out.threads_cols = TC;
    if (job_image) job_image->clear();
    if (job_is_col) job_is_col->clear();
    out.jobs.reserve(2 * count);

    std::vector<uint32_t> order(count);
    std::iota(order.begin(), order.end(), 0u);
    std::vector<double> work(count);
    for (size_t i = 0; i < count; ++i)
        work[i] = (double)compute_m(entries[i].width) * entries[i].height +
                  (double)compute_m(entries[i].height) * entries[i].width;
    std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t c) { return work[a] > work[c]; });

    std::vector<TileGroup> groups;  // an image's one or two next to each other
    groups.reserve(2 * count);
    std::vector<std::shared_ptr<const LinePlan>> plans(2 * count);  // rows, columns of every entry
    for (size_t i = 0; i < count; ++i) {
        plans[2 * i] = ctx.line_plan((int)entries[i].width, false);
        plans[2 * i + 1] = ctx.line_plan((int)entries[i].height, true);
    }
    out.hold_cols = column_kernel(TC, ctx.cu_count(), entries, count, plans);
    if (out.hold_cols == BATCH_ALL) TC = out.threads_cols = BATCH_THREADS;
    uint32_t counter = 0;
    uint64_t nitems = 0;
    for (uint32_t idx : order) {
        const BatchEntry& e = entries[idx];
        const int w = (int)e.width, h = (int)e.height;
        const LinePlan *rp = plans[2 * idx].get(), *cp = plans[2 * idx + 1].get();
        const int lpw_r = w > 1 ? lines_per_tile(*rp) : 0;
        const bool whole = runs_whole(w, h, *rp, *cp);
        // column tiles of images with a row pass run in the column phase (TC
        // threads); a single-column-pass image (w == 1) runs with the rows
        const int lpw_c = h <= 1             ? 0
                          : w > 1 && !whole ? lines_per_tile(TC, out.hold_cols, *cp)
                                            : lines_per_tile(*cp);
        const int ntr = w > 1 ? (h + lpw_r - 1) / lpw_r : 0;
        const int ntc = h > 1 ? (w + lpw_c - 1) / lpw_c : 0;
        const int sig = (dependent && w > 1 && h > 1 && !whole) ? (int)counter++ : -1;
        int rj = -1, cj = -1;
        if (w > 1) {
            BatchJob j{};
            j.job = ctx.make_job(*rp, e.src, e.dst, 1, w, h, e.inverse);
            j.shape = rp->shape;
            j.blue = rp->blue;
            j.cols = 0;
            j.ntiles = ntr;
            j.dep = -1;
            j.sig = sig;
            rj = (int)out.jobs.size();
            out.jobs.push_back(j);
            if (job_image) job_image->push_back(idx);
            if (job_is_col) job_is_col->push_back(0);
        }
        if (h > 1) {
            BatchJob j{};
            // the column pass reads the row pass's output when there is one
            j.job = ctx.make_job(*cp, w > 1 ? e.dst : e.src, e.dst, w, 1, w, e.inverse);
            j.shape = cp->shape;
            j.blue = cp->blue;
            j.cols = 1;
            j.ntiles = ntc;
            j.dep = sig;
            j.dep_need = ntr;
            j.sig = -1;
            cj = (int)out.jobs.size();
            out.jobs.push_back(j);
            if (job_image) job_image->push_back(idx);
            if (job_is_col) job_is_col->push_back(1);
        }
        auto add = [&](int phase, int kind, const LinePlan& lp, int lines, int job, uint32_t first, int tiles) {
            const double cost = lines * line_cost(lp) * (lp.blue ? 2 : 1) * (kind == 0 ? 2 : 1);
            groups.push_back({phase, lp.m, lp.shape, lp.blue, kind, (uint32_t)job, first, (uint32_t)tiles,
                              std::max<int64_t>(1, std::llround(cost))});
            nitems += (uint64_t)tiles;
        };
        if (whole) {
            add(1, 0, *rp, lpw_r, rj, BATCH_WHOLE | (uint32_t)cj, 1);
        } else {
            if (ntr > 0) add(1, 1, *rp, lpw_r, rj, 0, ntr);
            if (ntc > 0) add(w > 1 ? 2 : 1, 2, *cp, lpw_c, cj, 0, ntc);
        }
    }
    out.keep = std::move(plans);
    if (nitems > 0x7fffffff) throw Error(MDFT_ERR_SIZE, "batch of " + std::to_string(nitems) + " tiles");
    out.items.resize((size_t)nitems);
    uint32_t* words = reinterpret_cast<uint32_t*>(out.items.data());
    if (dependent) {
        // rows of image k+1 before columns of image k: a column tile only
        // waits on row tiles with smaller tickets
        const TileGroup* late = nullptr;  // columns of the image before
        for (const TileGroup& g : groups) {
            if (g.kind != 2) {
                words = write_tiles(g, words);
                if (late) words = write_tiles(*late, words);
                late = nullptr;
                continue;
            }
            if (late) words = write_tiles(*late, words);
            late = &g;
        }
        if (late) write_tiles(*late, words);
        out.nphase1 = (uint32_t)nitems;
    } else {
        out.nphase1 = lay_out_tiles(groups, words);
    }
    out.ncounters = counter;
}

// Workgroups of a launch are dealt to the XCDs round-robin: block b runs on
// XCD b % 8, and each XCD has its own L2.  Give every job (its tiles, and
// with them its chirp, diagonal and twiddle tables and, for column tiles,
// the cache lines neighbouring tiles share) to one XCD, balancing the XCDs'
// total cost (largest run first, jobs larger than a sixteenth of the launch
// split), then lay the eight queues out so that queue x fills the blocks
// b % 8 == x.  Within a queue the order of the groups is kept.  Only the last
// step touches single tiles: a burst of requests makes thousands, and its launch
// waits for them (15 requests of 4781 tiles: 17 us for the whole build on the
// scheduler's thread, 115 with every tile sorted, costed and copied by itself).
static uint32_t* arrange_for_xcds(const TileGroup* groups, size_t ngroups, uint32_t* words)
{
    constexpr int NXCD = 8;
    int64_t total = 0;
    size_t n = 0;
    for (size_t i = 0; i < ngroups; ++i) {
        total += groups[i].cost * groups[i].count;
        n += groups[i].count;
    }
    struct Run {
        uint32_t job, first, count;
        int64_t cost;
    };
    std::vector<Run> runs;
    for (size_t i = 0; i < ngroups; ++i) {
        const TileGroup& g = groups[i];
        const int64_t most = std::max<int64_t>(1, total / (2 * NXCD * g.cost));
        for (uint32_t t = 0; t < g.count;) {
            const uint32_t k = (uint32_t)std::min<int64_t>(most, g.count - t);
            runs.push_back({g.job, g.first + t, k, g.cost * k});
            t += k;
        }
    }
    std::vector<uint32_t> by_cost(runs.size());
    std::iota(by_cost.begin(), by_cost.end(), 0u);
    std::stable_sort(by_cost.begin(), by_cost.end(), [&](uint32_t a, uint32_t c) { return runs[a].cost > runs[c].cost; });
    std::vector<uint8_t> owner(runs.size());
    int64_t load[NXCD] = {};
    for (uint32_t r : by_cost) {
        int best = 0;
        for (int x = 1; x < NXCD; ++x)
            if (load[x] < load[best]) best = x;
        owner[r] = (uint8_t)best;
        load[best] += runs[r].cost;
    }
    struct Queue {
        std::vector<Run> runs;
        size_t at = 0, left = 0;  // the run being read, tiles not yet placed
    } queue[NXCD];
    for (size_t r = 0; r < runs.size(); ++r) {
        queue[owner[r]].runs.push_back(runs[r]);
        queue[owner[r]].left += runs[r].count;
    }
    // while no queue is dry, queue x fills the blocks x, x + 8, ..
    size_t rounds = queue[0].left;
    for (const Queue& q : queue) rounds = std::min(rounds, q.left);
    for (int x = 0; x < NXCD; ++x) {
        Queue& q = queue[x];
        uint32_t* w = words + 2 * x;
        for (size_t left = rounds; left > 0;) {
            Run& r = q.runs[q.at];
            const uint32_t job = r.job, first = r.first, k = (uint32_t)std::min<size_t>(left, r.count);
            for (uint32_t t = 0; t < k; ++t, w += 2 * NXCD) w[0] = job, w[1] = first + t;
            r.first += k, r.count -= k, left -= k;
            q.at += r.count == 0;
        }
        q.left -= rounds;
    }
    words += 2 * NXCD * rounds;
    // then its slots take the longest remaining queue's items
    for (size_t b = NXCD * rounds; b < n; ++b) {
        int x = int(b % NXCD);  // block index within this launch
        if (queue[x].left == 0)
            for (int y = 0; y < NXCD; ++y)
                if (queue[y].left > queue[x].left) x = y;
        Queue& q = queue[x];
        Run& r = q.runs[q.at];
        *words++ = r.job;
        *words++ = r.first++;
        q.at += --r.count == 0;
        --q.left;
    }
    return words;
}

uint32_t lay_out_tiles(std::vector<TileGroup>& groups, uint32_t* words)
{
    std::stable_sort(groups.begin(), groups.end(), [](const TileGroup& a, const TileGroup& c) {
        return std::make_tuple(a.phase, -a.m, a.shape, a.blue, a.kind) <
               std::make_tuple(c.phase, -c.m, c.shape, c.blue, c.kind);
    });
    size_t n1 = 0;
    uint32_t tiles1 = 0;
    for (; n1 < groups.size() && groups[n1].phase == 1; ++n1) tiles1 += groups[n1].count;
    words = arrange_for_xcds(groups.data(), n1, words);
    arrange_for_xcds(groups.data() + n1, groups.size() - n1, words);
    return tiles1;
}

}  // namespace mdft
