// gemm_split.hpp — the k partitions of a product, and the tile for them, from
// a model of the device time of a product on a tile. Host code only.
//
// Products with few output tiles against the 256 CUs walk a long serial k
// loop on a mostly idle chip; partitions shorten the loop and cost a pass over
// the partial outputs.
#pragma once

#include "internal.hpp"

#include <algorithm>
#include <cmath>

namespace blis_amd {

// The k partitions for a shape, and the tile the model found fastest (-1:
// none looked for).
struct SplitChoice {
    int split = 1;
    int tile = -1;
};

// A product on one tile with `parts` k partitions takes, in us: a workgroup's
// launch, prologue and epilogue (fixed), and its serial chain of k slabs. A slab
// is bound by its own latency (slab), stretched once more workgroups are
// launched than fit the chip (`resident` per CU), and by the CU's matrix
// cores (full per workgroup on the CU; no less than 2 bm bn bk flops at the
// card's peak, 78.6 and 157.3 TFLOP/s over 256 CUs). The two overlap in part:
// their hypotenuse fits better than the larger of them. For parts > 1 the
// reduction follows: its launch, a chain of `parts` additions, and one pass over the
// partitions.
struct TileCost {
    int tile, bm, bn, bk, resident;
    double slab, full, fixed;
};
struct SplitModel {
    int tiles;
    TileCost t[4];
    double reduce, reduce_part, rate;   // us, us per partition, bytes per us
    // Masked products (gemmt, syrk) launch workgroups for all tiles, and those
    // of the tiles that are not stored end at once, which loads the CUs
    // unevenly: a CU's matrix cores serve this many workgroups more than an
    // even spread of the others gives it (which hides the 64 x 64 tiles' latency).
    double uneven;
    // Bytes per us at which all workgroups together read their operands (masked
    // products over a deep k; no bound in sight for plain ones).
    double operands;
};

// Fitted to the device times on these tiles with 1 to 64 partitions of 264 GEMM
// and 98 SYRK shapes per type (m, n in [32, 8192], k in [128, 16384], SYRK to
// 65536, each operand in both layouts): rms error 8% and 9% over 7,500 FP64
// and 8,100 FP32 timings of GEMM, 10% and 13% for SYRK. The pair it picks is
// within 2.4%, 3.1%, 3.0% and 5.2% of the best timing in geometric mean. A fit
// without the floor under `full` had given the 32 x 32 FP64 tile no throughput
// limit, which sent every split product to it: 12% (GEMM) and 14% (SYRK)
// from the best, 1024 x 1024 x 8192 at 404 us in place of 281.
inline const SplitModel& split_model(Dt dt, bool masked) {
    static const SplitModel plain64 = { 4, {
        { 3, 64, 64, 16, 4, 0.698, 0.483, 4.4 },
        { 4, 32, 32, 16, 8, 0.420, 0.147, 4.7 },
        { 10, 64, 128, 16, 3, 0.620, 0.931, 5.9 },
        { 6, 128, 128, 16, 2, 1.020, 1.783, 6.4 } }, 0.5, 0.18, 6.5e6, 0.0, 0.0 };
    static const SplitModel plain32 = { 4, {
        { 3, 64, 64, 32, 4, 0.929, 0.473, 4.3 },
        { 4, 32, 32, 32, 8, 0.468, 0.176, 4.2 },
        { 9, 128, 64, 32, 3, 1.096, 0.925, 4.6 },
        { 10, 64, 128, 32, 3, 1.117, 0.911, 5.1 } }, 2.0, 0.255, 6.3e6, 0.0, 0.0 };
    static const SplitModel masked64 = { 2, {
        { 3, 64, 64, 16, 4, 0.094, 0.533, 3.2 },
        { 4, 32, 32, 16, 8, 0.342, 0.165, 2.2 } }, 3.0, 0.20, 9.6e6, 1.19, 10.5e6 };
    static const SplitModel masked32 = { 2, {
        { 3, 64, 64, 32, 4, 0.0, 0.532, 3.4 },
        { 4, 32, 32, 32, 8, 0.322, 0.200, 2.1 } }, 3.3, 0.33, 6.3e6, 1.59, 9.8e6 };
    return dt == Dt::F64 ? (masked ? masked64 : plain64) : (masked ? masked32 : plain32);
}

inline double split_cost(Dt dt, const SplitModel& sm, const TileCost& t, int64_t m, int64_t n,
                         int64_t k, int parts, bool masked) {
    const int64_t gm = (m + t.bm - 1) / t.bm, gn = (n + t.bn - 1) / t.bn;
    const double tiles = masked ? 0.5 * (double)(gm * gn + std::max(gm, gn)) : (double)(gm * gn);
    // As split_params cuts it: whole 64-deep blocks.
    const int64_t blocks = (k + 63) / 64, chunk = (blocks + parts - 1) / parts * 64;
    parts = (int)((k + chunk - 1) / chunk);
    const double slabs = (double)((std::min(chunk, k) + t.bk - 1) / t.bk);
    const double wgs = tiles * parts, per_cu = std::ceil(wgs / 256.0);
    const bool fits = per_cu <= t.resident;
    const double lat = t.slab * (fits ? 1.0 : wgs / (256.0 * t.resident));
    const double thr = t.full * (masked ? 1.05 * wgs / 256.0 + sm.uneven
                                        : fits ? per_cu : wgs / 256.0 + 0.5);
    double us = slabs * std::hypot(lat, thr);
    if (sm.operands > 0.0)
        us = std::max(us, tiles * (t.bm + t.bn) * (double)k * (double)dt_size(dt) / sm.operands);
    us += t.fixed;
    if (parts > 1) {
        const double bytes = (2.0 * parts + 2.0) * (double)m * (double)n * (double)dt_size(dt);
        us += sm.reduce + sm.reduce_part * parts + (masked ? 0.6 : 1.0) * bytes / sm.rate;
    }
    return us;
}

// The pair of partitions (at most `most`) and tile with the least modelled
// time. The partitions depend on the type, k and the pair of m and n in either
// order, so every tile and every operand layout gives the same bits: a product
// whose C is stored by rows is computed transposed (layout(), gemm_plan.hpp).
// One pass stays: up to k = 512 (single calls and batches of such products
// agree bit for bit), where the partitions would take over 48 MiB, and from
// 2048 stored tiles of 64 x 64, which fill the chip by themselves. An output of
// a single 64 x 64 tile keeps partitions of 1024, up to 64 of them. A masked
// FP32 product of k < 128, which no fitted shape has, keeps the size heuristic's
// tile, whose 64-row waves write C in vectors (n = 3452, k = 28: 28 us, 40 on
// 64 x 64).
inline SplitChoice gemm_choose_split(Dt dt, int64_t m, int64_t n, int64_t k, bool masked,
                                     int most = 64) {
    SplitChoice c;
    const int64_t t64 = ((m + 63) / 64) * ((n + 63) / 64);
    if ((masked ? t64 / 2 : t64) >= 2048) return c;
    if (masked ? dt == Dt::F32 && k < 128 : k <= 512) return c;
    if (t64 == 1 && !masked) {
        if (k >= 2048) c.split = (int)std::min<int64_t>({ k / 1024, 64, most });
        c.tile = 4;
        return c;
    }
    static const int parts[] = { 1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32, 48, 64 };
    const SplitModel& sm = split_model(dt, masked);
    double best = 0.0;
    const int64_t hi = std::max(m, n), lo = std::min(m, n);
    for (int s : parts) {
        if (s > 1 && (k <= 512 || s > most || s * 64 > k ||
                      (double)s * m * n * dt_size(dt) > 48.0 * (1 << 20)))
            break;
        for (int q = 0; q < sm.tiles; ++q) {
            const double us = split_cost(dt, sm, sm.t[q], hi, lo, k, s, masked);
            if (best == 0.0 || us < best) { best = us; c.split = s; }
        }
    }
    // The tile for these partitions, from m and n as they are.
    best = 0.0;
    for (int q = 0; q < sm.tiles; ++q) {
        const double us = split_cost(dt, sm, sm.t[q], m, n, k, c.split, masked);
        if (best == 0.0 || us < best) { best = us; c.tile = sm.t[q].tile; }
    }
    return c;
}

} // namespace blis_amd
