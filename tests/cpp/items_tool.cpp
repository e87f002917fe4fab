// Lays out random batches with the library (lay_out_tiles) and tile by tile as
// the rule reads, and compares the items.  Prints "equal <batches> <tiles>" and
// the time of each way for the last batch, or the first difference.
#include <algorithm>
#include <chrono>
#include <cstdint>
#include <cstdio>
#include <numeric>
#include <random>
#include <tuple>
#include <utility>
#include <vector>

// from math_amd/csrc/host/batch_builder.hpp, without the HIP headers it needs
namespace mdft {
struct TileGroup {
    int phase;
    int m, shape, blue, kind;
    uint32_t job, first, count;
    int64_t cost;
};
uint32_t lay_out_tiles(std::vector<TileGroup>& groups, uint32_t* words);
}  // namespace mdft

using mdft::TileGroup;
using Item = std::pair<uint32_t, uint32_t>;

namespace {

struct Tile {
    TileGroup g;
    uint32_t seq;
    Item v;
};

// runs of consecutive tiles of a job up to a sixteenth of the cost, the dearest first to the least loaded XCD
void arrange(const std::vector<Tile>& tiles, std::vector<Item>& out)
{
    const size_t n = tiles.size();
    double total = 0;
    for (const Tile& t : tiles) total += (double)t.g.cost;
    struct Run {
        size_t begin, end;
        double cost;
    };
    std::vector<Run> runs;
    for (size_t i = 0; i < n;) {
        size_t j = i;
        double c = 0;
        while (j < n && tiles[j].v.first == tiles[i].v.first && (j == i || c + (double)tiles[j].g.cost <= total / 16))
            c += (double)tiles[j++].g.cost;
        runs.push_back({i, j, c});
        i = j;
    }
    std::vector<size_t> by_cost(runs.size());
    std::iota(by_cost.begin(), by_cost.end(), size_t(0));
    std::stable_sort(by_cost.begin(), by_cost.end(), [&](size_t a, size_t b) { return runs[a].cost > runs[b].cost; });
    std::vector<int> owner(runs.size());
    double load[8] = {};
    for (size_t r : by_cost) {
        const int best = int(std::min_element(load, load + 8) - load);
        owner[r] = best;
        load[best] += runs[r].cost;
    }
    std::vector<Item> queue[8];
    for (size_t r = 0; r < runs.size(); ++r)
        for (size_t i = runs[r].begin; i < runs[r].end; ++i) queue[owner[r]].push_back(tiles[i].v);
    size_t pos[8] = {};
    for (size_t b = 0; b < n; ++b) {
        int x = int(b % 8);
        if (pos[x] == queue[x].size()) {
            size_t most = 0;
            for (int y = 0; y < 8; ++y)
                if (queue[y].size() - pos[y] > most) most = queue[y].size() - pos[y], x = y;
        }
        out.push_back(queue[x][pos[x]++]);
    }
}

uint32_t tile_by_tile(const std::vector<TileGroup>& groups, std::vector<Item>& out)
{
    std::vector<Tile> tiles;
    uint32_t seq = 0;
    for (const TileGroup& g : groups)
        for (uint32_t t = 0; t < g.count; ++t) tiles.push_back({g, seq++, {g.job, g.first + t}});
    std::stable_sort(tiles.begin(), tiles.end(), [](const Tile& a, const Tile& c) {
        return std::make_tuple(a.g.phase, -a.g.m, a.g.shape, a.g.blue, a.g.kind, a.seq) <
               std::make_tuple(c.g.phase, -c.g.m, c.g.shape, c.g.blue, c.g.kind, c.seq);
    });
    const auto p2 = std::find_if(tiles.begin(), tiles.end(), [](const Tile& t) { return t.g.phase == 2; });
    arrange({tiles.begin(), p2}, out);
    arrange({p2, tiles.end()}, out);
    return (uint32_t)(p2 - tiles.begin());
}

double us(std::chrono::steady_clock::time_point a, std::chrono::steady_clock::time_point b)
{
    return std::chrono::duration<double, std::micro>(b - a).count();
}

}  // namespace

int main()
{
    std::mt19937 rng(7);
    size_t total = 0;
    double t_lib = 0, t_ref = 0;
    const int batches = 400;
    for (int k = 0; k < batches; ++k) {
        // images of random geometry; the last batch is a burst of 16 large ones
        const bool burst = k + 1 == batches;
        const uint32_t images = burst ? 16 : rng() % 40;
        std::vector<TileGroup> groups;
        uint32_t job = 0, tiles = 0;
        for (uint32_t i = 0; i < images; ++i) {
            const int m = (rng() % 2 ? 1 : 3) << (5 + rng() % 8), shape = (int)(rng() % 20), blue = (int)(rng() % 2);
            const int64_t cost = 1 + rng() % (rng() % 4 ? 9 : 400000);
            if (!burst && rng() % 4 == 0) {
                groups.push_back({1, m, shape, blue, 0, job, 0x80000000u | (job + 1), 1, cost});
                job += 2, tiles += 1;
                continue;
            }
            const uint32_t rows = burst ? 250 : rng() % 5 ? 1 + rng() % 90 : 0, cols = burst ? 60 : rng() % 90;
            if (rows) groups.push_back({1, m, shape, blue, 1, job++, 0, rows, cost});
            if (cols) groups.push_back({rows ? 2 : 1, m, shape, 1 - blue, 2, job++, 0, cols, cost * 2});
            tiles += rows + cols;
        }
        std::vector<Item> want;
        std::vector<uint32_t> words(2 * (size_t)tiles + 2, 0xdeadbeefu);
        const auto a = std::chrono::steady_clock::now();
        const uint32_t n1 = tile_by_tile(groups, want);
        const auto b = std::chrono::steady_clock::now();
        const uint32_t g1 = mdft::lay_out_tiles(groups, words.data());
        const auto c = std::chrono::steady_clock::now();
        t_ref = us(a, b), t_lib = us(b, c);
        if (n1 != g1 || words[2 * (size_t)tiles] != 0xdeadbeefu) {
            std::printf("batch %d: %u items of phase 1, expected %u\n", k, g1, n1);
            return 1;
        }
        for (size_t i = 0; i < want.size(); ++i)
            if (words[2 * i] != want[i].first || words[2 * i + 1] != want[i].second) {
                std::printf("batch %d item %zu: (%u, %x), expected (%u, %x)\n", k, i, words[2 * i], words[2 * i + 1],
                            want[i].first, want[i].second);
                return 1;
            }
        total += want.size();
    }
    std::printf("equal %d %zu\nlibrary %.1f us, tile by tile %.1f us\n", batches, total, t_lib, t_ref);
    return 0;
}
