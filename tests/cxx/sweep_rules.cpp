// The host rules of the SpMM sweep kernel over sizes drawn at random: what the kernel and its launch take for granted.
#include "../../library_amd/csrc/asx_internal.hpp"

#include <cmath>
#include <cstdio>
#include <random>

using namespace asx;

static bool launched(const SpmmSweep &sw)  // the kernel is instantiated for it
{
    const int most = sw.log_lanes == 3 ? 8 : sw.log_lanes == 4 ? 16 : 20;
    return sw.log_lanes >= 3 && sw.log_lanes <= 6 && sw.slots >= 4 && sw.slots <= most && sw.slots % 4 == 0;
}

int main()
{
    std::mt19937_64 gen(7);
    const auto log_uniform = [&](double lo, double hi) { return std::exp(std::uniform_real_distribution<double>(std::log(lo), std::log(hi))(gen)); };
    long taken = 0, asked = 0, several = 0;
#define REQUIRE(what)                                                                                                           \
    if (!(what)) {                                                                                                              \
        std::printf("%s: m %d n %d nnz %d ncols %d sv %zu groups %d longest %lld\n", #what, m, n, nnz, ncols, sv, t.groups,     \
                    (long long)longest);                                                                                        \
        return 1;                                                                                                               \
    }
    for (int turn = 0; turn < 400000; ++turn) {
        const size_t sv = gen() % 2 ? 4 : 8;
        const int32_t m = (int32_t)log_uniform(1, 2e7), n = (int32_t)log_uniform(1, 2e7);
        const int32_t nnz = (int32_t)std::min(2e9, m * log_uniform(1, 2000));
        const int32_t ncols = gen() % 3 ? (int32_t)log_uniform(1, 3000) : 32 * (int32_t)log_uniform(1, 40);
        const int tile_bytes[] = {128, 256, 512, 1024};
        const SpmmTiling t = spmm_tiling(ncols, tile_bytes[gen() % 4], sv);
        const int32_t items = spmm_segment_items(m, nnz, ncols, sv);
        for (int planned = 0; planned < 2; ++planned) {
            const bool chunked = planned && gen() % 2;
            const int64_t longest = planned ? nnz / m + (int64_t)log_uniform(1, 100) : spmm_sweep_ask_longest(m, nnz, t.groups);
            const int chains = spmm_sweep_chains(longest, t.groups, chunked);
            REQUIRE(chains == 0 || chains == 1 || ((chains == 2 || chains == 4) && chains == t.groups));
            // as many sums as the row-ordered kernels have, or few enough elements for one
            REQUIRE(chains != 1 || longest <= (chunked ? std::min(spmm_dealt(t.groups), kChunkWideLeast) : spmm_dealt(t.groups)));
            REQUIRE(chains < 2 || !chunked || longest <= kChunkWideLeast);
            const SpmmSweep sw = spmm_sweep(m, n, nnz, ncols, sv, chains);
            if (sw.slots == 0) continue;
            ++taken;
            several += chains > 1;
            const int groups = kWave >> sw.log_lanes;
            REQUIRE(chains >= 1 && launched(sw) && sw.slots <= 1 << sw.log_lanes && sw.rows >= 1 && sw.rows * chains <= sw.slots && sw.slots % chains == 0);
            REQUIRE(sw.chains == chains && (chains == 1 || (spmm_dealt(chains) == spmm_dealt(4) && sw.log_lanes >= 4)) && sw.rows < 256);
            REQUIRE(sw.cap >= 2 && sw.cap % 2 == 0 && sw.cap <= spmm_sweep_cap(sv));
            REQUIRE(4 * (std::min(sw.cap, spmm_sweep_cap(sv) - 2) * (sv + 4) * (kBlock / kWave) + 32) <= 160 * 1024);
            REQUIRE(sw.tiles >= 1 && sw.tiles <= 65535 && ncols / sw.tiles >= (int64_t)(16 / sv));
            REQUIRE(ceil_div64(ncols, sw.tiles) <= (int64_t)(16 / sv) << sw.log_lanes);
            const int64_t blocks = spmm_sweep_blocks(sw, m);
            REQUIRE(blocks % kXcds == 0 && blocks * (kBlock / kWave) * sw.rows * groups >= m);
            REQUIRE(sw.width >= 1);
            if (planned || !spmm_sweep_askable(spmm_sweep_shape(m, nnz, ncols, sv, 1), m, nnz, ncols, sv, items)) continue;
            ++asked;
            REQUIRE(longest <= items && spmm_segments(m, nnz, items) >= 2);  // whole rows only, and splits to look for
            REQUIRE(spmm_sweep_ask_blocks(chains) <= kSweepAskBlocks);
            REQUIRE(t.log_lanes >= 3 && t.vec == (int)(16 / sv));  // the merge kernel has a variant that looks at the answer
        }
    }
    std::printf("taken %ld, several sums %ld, asked %ld\n", taken, several, asked);
    return taken > 1000 && several > 100 && asked > 100 ? 0 : 1;
}
