// Plan and launch of the few-rows projection (gemm_rows.hpp).
#include <algorithm>

#include "gemm_rows.hpp"

namespace fh {

namespace {

// What one super-block of one weight tile costs a wave, in us, with two waves on the SIMD: the decode,
// the matrix instructions of 16 or 32 rows and their share of the stream.  From 17408 x 5120 and
// 5120 x 17408 (f16: 17.7 / 21.2 us at 16 / 32 rows for Q4_K, 30.8 / 40.5 for Q6_K).  f32 rows count 2.3 in every
// format here, as measured on Q4_K before their sums were paired: it places tiles and segments only (whether the
// kernel takes the call is f32_rows_pay's, with the present 2.6 to 3.0; 16 rows of 17408 x 5120 take 46 us for Q4_K,
// 60 for Q6_K), and a row's sums follow from that placement.
double unit_us(uint32_t ggml_type, uint32_t x_dtype, uint32_t rows) {
    if (x_dtype == FH_F32) return 2.3;
    switch (ggml_type) {
        case kQ4K: return rows == 16 ? 0.90 : 1.15;
        case kQ6K: return rows == 16 ? 1.80 : 2.40;
        default: return rows == 16 ? 1.30 : 1.70;
    }
}

constexpr double kStartUs = 4.0;      // launch, first loads, exchange of the waves' sums
constexpr double kExchangeUs = 4.0;   // partial sums of K segments through device memory

constexpr uint32_t kMostWorkgroups = 1u << 22;   // of a launch, and half of what a grid of 512 threads each may have

}  // namespace

RowsPlan gemm_rows_plan(uint32_t ggml_type, uint32_t n, uint32_t k, uint32_t m, uint32_t x_dtype, int cu_count) {
    RowsPlan plan{};
    const uint32_t nb = k / 256, tiles = (n + 15) / 16, cus = cu_count > 0 ? (uint32_t)cu_count : 256u;
    plan.rows = x_dtype != FH_F32 && m > 16 ? 32 : 16;
    plan.k_waves = nb >= 8 ? 8 : nb >= 4 ? 4 : nb >= 2 ? 2 : 1;
    const uint32_t tile_waves = 8 / plan.k_waves;
    const double unit = unit_us(ggml_type, x_dtype, 16);
    // Tiles per wave and K segments, from the matrix alone: the sums of a row then do not depend on how
    // many rows come with it.  Rounds of one workgroup per compute unit, each as long as the
    // super-blocks of its longest wave.  8 x 17408 x 5120: 17.2 us with five tiles in one round of 218
    // workgroups, 21 - 26 with fewer tiles in more rounds, 25 - 31 with K cut in two; 8 x 5120 x 17408:
    // 20.8 with four tiles and three segments, 22 - 41 without segments.
    double best = 1e300;
    for (uint32_t segments = 1; segments <= 8; ++segments) {
        const uint32_t seg_blocks = (nb + segments - 1) / segments;
        if ((nb + seg_blocks - 1) / seg_blocks != segments || (segments > 1 && seg_blocks < plan.k_waves)) continue;
        const uint32_t per_wave = (seg_blocks + plan.k_waves - 1) / plan.k_waves;
        for (uint32_t t = 1; t <= 5; ++t) {
            const uint32_t tile_groups = (tiles + t * tile_waves - 1) / (t * tile_waves);
            const uint64_t wgs = (uint64_t)tile_groups * segments;
            const double us = (double)((wgs + cus - 1) / cus) * (kStartUs + per_wave * t * unit) +
                              (segments > 1 ? kExchangeUs : 0.0);
            if (us < best) {
                best = us;
                plan.tiles = t;
                plan.segments = segments;
                plan.seg_blocks = seg_blocks;
                plan.tile_groups = tile_groups;
            }
        }
    }
    const uint32_t per_wave = (plan.seg_blocks + plan.k_waves - 1) / plan.k_waves;
    // A batch whose partial sums exceed the scratch a device has at all times, or whose tiles the counters or
    // the grid, runs in several launches: no batch makes the scratch grow (8192 rows of 5120 x 17408 would ask for
    // 480 MiB), and one launch's rows, 272 there, are sixteen rounds of the chip.
    uint64_t most = kMostWorkgroups / ((plan.tile_groups + 7) / 8 * 8);   // row groups
    if (plan.segments > 1) {
        most = std::min<uint64_t>(most, fh_device::kScratchFloor / ((uint64_t)plan.segments * n * sizeof(float) * plan.rows));
        most = std::min<uint64_t>(most, fh_device::kCounterWords / plan.tile_groups);
    }
    plan.run_rows = (uint32_t)std::min<uint64_t>(m, std::max<uint64_t>(most, 1) * plan.rows);
    // (from two rounds on a compute unit's next workgroup starts as soon as one ends: rounds need not be whole,
    // except that up to 16 rows, whose workgroups mostly wait for weights of their own, the second costs more than
    // the first and the third is whole: 8 x 28672 x 4096 in two rounds takes 26.5 us for Q4_K and 36 for Q5_K, the
    // rows-resident kernel 24 and 33; 32 x 34816 x 5120 42 for Q4_K, that kernel 50)
    const uint64_t groups = ((uint64_t)m + plan.rows - 1) / plan.rows;
    const double rounds = (double)(plan.tile_groups * plan.segments * groups) / (double)cus;
    const bool waits = m <= 16 && x_dtype != FH_F32;
    const double counted = rounds <= 1.0   ? 1.0
                           : rounds <= 2.0 ? (waits ? 2.3 : 2.0)
                                           : std::max(rounds + 0.2, waits ? 3.0 : 0.0);
    plan.estimate_us = counted * (kStartUs + per_wave * plan.tiles * unit_us(ggml_type, x_dtype, plan.rows)) +
                       (plan.segments > 1 ? kExchangeUs : 0.0);
    if (plan.rows == 32 && m > 32) {
        // several groups share the weights in an L2 and the longest and shortest waves a SIMD: fitted to the 385 plans of
        // 40 - 128 rows in profiles/few_rows_against_tiles_us.txt (eleven shapes, five formats), 8% in the mean square (Q6_K's decode of four
        // and five tiles is above the fit)
        const double tile = ggml_type == kQ4K     ? 1.39
                            : ggml_type == kQ5K   ? 1.88
                            : ggml_type == kQ6K   ? 2.34
                            : ggml_type == kIQ4XS ? 1.55
                                                  : 1.77;
        // (of waves with one or two super-blocks the longer ones count for three tenths, where there are more the mean does: IQ4_XS 67
        // x 13035 x 3328, 13 in eight waves, was put at 33 us by the mean; it takes 42, the tiles 33, and Q8_0 102 x 2271 x 2816 16.4,
        // on the resident kernel 13.9.  Of the products in profiles/routes_us.txt 22 take 5% longer than by the estimates before
        // this fit, by the mean alone 38, with three tenths everywhere 18, but twice as many others lose by it.)
        const double mean = (double)plan.seg_blocks / plan.k_waves, share = per_wave > 2 ? mean : mean + 0.3 * (per_wave - mean);
        const double fitted = 2.3 + (rounds <= 1.0 ? 1.0 : std::max(1.84, rounds)) * (1.9 + share * (0.35 + plan.tiles) * tile) +
                              (plan.segments > 1 ? 5.5 : 0.0);
        plan.estimate_us = ggml_type == kQ6K ? std::max(plan.estimate_us, fitted) : std::min(plan.estimate_us, fitted);
    }
    plan.groups = (plan.run_rows + plan.rows - 1) / plan.rows;
    plan.counters = plan.segments > 1 ? (size_t)plan.tile_groups * plan.groups : 0;
    plan.partial_bytes = plan.segments > 1 ? (size_t)plan.segments * plan.run_rows * n * sizeof(float) : 0;
    return plan;
}

// A batch of exact f32 rows.  The GEMV reads every weight once per row, but with few rows and small matrices its
// workgroups fill a chip that one launch of this kernel leaves idle.  Q4_K and Q5_K take the faster of the two by
// estimate, fitted to 4 - 48 rows of fifteen shapes from 256 x 256 to 151936 x 2048 and within 5% of the faster one
// in all but three of 196 measurements, the worst 14% (four Q5_K rows of 151936 x 2048; us, GEMV against this kernel: 16 x 256 x 256 Q5_K 3.7 / 6.8,
// 8 x 1024 x 4096 7.4 / 11.6 and 16 rows 10.6 / 11.7, 4 / 8 / 16 x 5120 x 5120 17.8 / 29.7 / 54.0 against 21.0).  Both
// are 1.0e-7 (rel-L2) from 64 bits there.  For the other formats the GEMV is at 1.8e-7 to 2.2e-7 and this kernel at
// 0.9e-7 to 1.2e-7, so they keep it also where the GEMV is faster (16 x 256 x 256 Q6_K 3.9 / 7.6, 8 x 1024 x 4096
// 8.1 / 12.3, even from 16 rows there and from four at 4096 x 4096).
bool f32_rows_pay(const RowsPlan& plan, uint32_t ggml_type, uint32_t n, uint32_t k, uint32_t m, int cu_count) {
    if (ggml_type != kQ4K && ggml_type != kQ5K) return true;
    if (m >= 6 && (uint64_t)n * (k / 256) >= 65536u) return true;   // (from 4096 x 4096 on without exception)
    // us per super-block: of a weight tile and wave here, per million of the matrix and per row there (rows of more
    // than 24 are cut into K segments, which meet in memory)
    const double unit = ggml_type == kQ4K ? 2.6 : 3.0;
    const double gemv_unit = (ggml_type == kQ4K ? 21.0 : 35.0) * (k > 24 * 256 ? 1.4 : 1.0);
    const uint32_t per_wave = (plan.seg_blocks + plan.k_waves - 1) / plan.k_waves;
    const uint64_t groups = ((uint64_t)m + plan.rows - 1) / plan.rows;
    const double rounds = (double)(plan.tile_groups * plan.segments * groups) / (double)(cu_count > 0 ? cu_count : 256);
    const double here = (rounds <= 1.0 ? 1.0 : rounds <= 2.0 ? 2.0 : rounds + 0.2) * (3.7 + per_wave * (0.9 + plan.tiles * unit));
    const double blocks = (double)m * (double)n * (double)(k / 256) * 1e-6;
    return here < 4.0 + std::max(0.0, blocks - 0.08) * gemv_unit;   // (80000 super-blocks run side by side)
}

void launch_gemm_rows(hipStream_t s, const GemmArgs& a) {
    const RowsPlan& plan = a.rows_plan;
    RowsParams p{};
    p.w = static_cast<const uint8_t*>(a.w);
    p.n = a.n;
    p.nb = a.k / 256;
    p.y_dtype = a.y_dtype;
    p.k_waves = plan.k_waves;
    p.tile_groups = plan.tile_groups;
    p.segments = plan.segments;
    p.seg_blocks = plan.seg_blocks;
    p.partials = a.partials;
    p.counters = a.counters;
    const size_t x_row = (size_t)a.k * dtype_bytes(a.x_dtype), y_row = (size_t)a.n * dtype_bytes(a.y_dtype);
    for (uint32_t first = 0; first < a.m; first += plan.run_rows) {
        p.x = static_cast<const uint8_t*>(a.x) + first * x_row;
        p.y = static_cast<uint8_t*>(a.y) + first * y_row;
        p.m = std::min(plan.run_rows, a.m - first);
        p.groups = (p.m + plan.rows - 1) / plan.rows;
        switch (a.ggml_type) {
            case kQ4K: launch_rows_q4_k(s, a.x_dtype, plan, p); break;
            case kQ5K: launch_rows_q5_k(s, a.x_dtype, plan, p); break;
            case kQ6K: launch_rows_q6_k(s, a.x_dtype, plan, p); break;
            case kIQ4XS: launch_rows_iq4_xs(s, a.x_dtype, plan, p); break;
            default: launch_rows_q8_0(s, a.x_dtype, plan, p); break;
        }
    }
}

}  // namespace fh
