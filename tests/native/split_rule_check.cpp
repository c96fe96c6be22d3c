// split_rule_check.cpp — the rule for k partitions (gemm_split.hpp) over random
// shapes, on the CPU: no modelled time lies below the card's peak, more than one
// tile is chosen, the partitions stay within their limits and are the same when
// m and n change places (C stored by rows or by columns). Prints "ok", or what went wrong.
#include "../../blis_amd/csrc/gemm_split.hpp"

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <set>

using namespace blis_amd;

static void fail(const char* what, Dt dt, int64_t m, int64_t n, int64_t k, bool masked) {
    std::printf("failed: %s (FP%d%s %lld x %lld x %lld)\n", what, dt == Dt::F64 ? 64 : 32,
                masked ? " masked" : "", (long long)m, (long long)n, (long long)k);
    std::exit(1);
}

int main() {
    std::mt19937_64 rng(1);
    auto size = [&](double lo, double hi) {
        return (int64_t)std::llround(std::exp(std::uniform_real_distribution<double>(
            std::log(lo), std::log(hi))(rng)));
    };
    for (Dt dt : { Dt::F64, Dt::F32 })
        for (bool masked : { false, true }) {
            const double peak = dt == Dt::F64 ? 78.6e6 : 157.3e6;   // flop per us
            const SplitModel& sm = split_model(dt, masked);
            std::set<int> split_tiles;
            for (int i = 0; i < 20000; ++i) {
                const int64_t m = size(16, 8192), n = masked ? m : size(16, 8192),
                              k = size(16, 65536);
                const double flops = (masked ? 1.0 : 2.0) * (double)m * n * k;
                for (int q = 0; q < sm.tiles; ++q)
                    for (int s : { 1, 2, 8, 64 })
                        if (split_cost(dt, sm, sm.t[q], m, n, k, s, masked) < flops / peak)
                            fail("faster than the peak", dt, m, n, k, masked);
                const SplitChoice c = gemm_choose_split(dt, m, n, k, masked);
                if (c.split < 1 || c.split > 64 || (c.split > 1 && k <= 512))
                    fail("partition count", dt, m, n, k, masked);
                if (c.split > 1 && m > 64 &&
                    (double)c.split * m * n * dt_size(dt) > 48.0 * (1 << 20))
                    fail("partitions over 48 MiB", dt, m, n, k, masked);
                if (gemm_choose_split(dt, n, m, k, masked).split != c.split)
                    fail("other partitions with m and n exchanged", dt, m, n, k, masked);
                if (gemm_choose_split(dt, m, n, k, masked, 1).split != 1)
                    fail("one pass asked for", dt, m, n, k, masked);
                if (c.split > 1) split_tiles.insert(c.tile);
            }
            if ((int)split_tiles.size() < 2) fail("one tile for every split", dt, 0, 0, 0, masked);
        }
    // Compute-bound over a deep k: large tiles, and partitions that fill the chip.
    for (int64_t k : { 4096, 8192, 16384 }) {
        const SplitChoice c = gemm_choose_split(Dt::F64, 1024, 1024, k, false);
        if (c.split < 2 || c.tile == 4) fail("deep k", Dt::F64, 1024, 1024, k, false);
    }
    std::printf("ok\n");
    return 0;
}
