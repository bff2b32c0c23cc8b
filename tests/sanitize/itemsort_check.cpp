// Checks nf::ItemSort (nf_internal.h), the counting sort of the work lists made
// on the host: every item of runs of varying length (tiles, tiles split over W
// source pencils, short tails) against a stable sort by key whose positions
// come from interleave_pos one by one.  Exit status 0 on success; the first
// failure is printed.
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <numeric>
#include <random>
#include <vector>

#include "nf_internal.h"

static bool same(const nf::WorkItem &a, const nf::WorkItem &b) {
    return a.sinkset == b.sinkset && a.first == b.first && a.nsink == b.nsink && a.kind_sic == b.kind_sic;
}

static int check(int tiles, int tails, int most, int keys, uint32_t seed) {
    std::mt19937 rng(seed);
    auto below = [&](int n) { return (int)(rng() % (uint32_t)n); };
    std::vector<nf::ItemRun> runs;
    for (int i = 0, t = tiles, q = tails; t + q > 0; i++) {
        if (below(t + q) < q) {  // a short tail
            runs.push_back({i, 64 * below(9), 64, 0, 1, 1, nf::kItemBuckets + below(keys)});
            runs.back().end = runs.back().first + 1 + below(nf::kTailLanes - 1);
            q--;
        } else {
            const int ny = below(3) ? 1 : 2 * below(3) + 1, step = ny > 1 ? 64 : 64 << below(3);
            runs.push_back({i, 0, step, 0, ny > 1 ? 3 : 2, ny, below(keys)});
            // Whole tiles, or the last one of fewer sinks.
            runs.back().end = step * (1 + below(most)) - (below(2) ? below(21) : 0);
            t--;
        }
    }
    std::vector<uint32_t> start(2 * nf::kItemBuckets + 1, 0u);
    nf::ItemSort sort{start.data()};
    for (const nf::ItemRun &r : runs) sort.add(r);
    const size_t n = sort.begin();
    std::vector<nf::WorkItem> got(n, nf::WorkItem{-1, 0, 0, 0});
    for (const nf::ItemRun &r : runs) sort.place(r, got.data());

    std::vector<std::pair<int, nf::WorkItem>> all;
    int64_t M = 0, T = 0;
    for (const nf::ItemRun &r : runs) {
        for (int f = r.first; f < r.end; f += r.step)
            for (int y = 0; y < r.ny; y++)
                all.push_back({r.key, {r.sinkset, f, std::min(r.step, r.end - f) + (r.ny > 1 ? 256 * y : 0), r.kind_sic}});
        (r.key < nf::kItemBuckets ? M : T) += r.count();
    }
    if (n != all.size() || (int64_t)n != M + T) {
        std::printf("seed %u: %zu items, %zu expected\n", seed, n, all.size());
        return 1;
    }
    std::stable_sort(all.begin(), all.end(), [](const auto &a, const auto &b) { return a.first < b.first; });
    for (int64_t i = 0; i < (int64_t)n; i++) {
        const bool tail = i >= M;
        const int64_t p = nf::interleave_pos(tail, tail ? i - M : i, M, T);
        if (!same(got[(size_t)p], all[(size_t)i].second)) {
            std::printf("seed %u (M %lld, T %lld): item %lld is not at position %lld\n", seed, (long long)M,
                        (long long)T, (long long)i, (long long)p);
            return 1;
        }
    }
    return 0;
}

int main() {
    int bad = 0;
    uint32_t seed = 1;
    for (int tiles = 0; tiles <= 40 && !bad; tiles++)
        for (int tails = 0; tails <= 120 && !bad; tails += 1 + tails / 8)
            for (int most : {1, 4, 40}) bad |= check(tiles, tails, most, 1 + (int)(seed % 37), seed), seed++;
    // A launch group's sizes: few tiles and many tails, and the other way round.
    const int big[][3] = {{200000, 10000, 12}, {3, 300000, 2}, {100000, 100000, 4}, {150000, 0, 9}, {0, 100000, 1}};
    for (const auto &b : big)
        if (!bad) bad |= check(b[0], b[1], b[2], nf::kItemBuckets, seed++);
    if (!bad) std::printf("ItemSort: every item at its interleaved position\n");
    return bad;
}
