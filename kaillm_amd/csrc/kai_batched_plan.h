// Launch plans of the batched GEMMs above 16 activation rows: which tile configuration, K split, tail
// of K pieces or second launch a product takes, from its type and shape alone (sized for the 256 CUs
// of an MI355X), and the scratch rule that callers query. Plain C++, so that a plan can be asked
// for without a device.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

#include "kai_formats.h"

namespace kai {

// ------------------------------------------------------------------------------ folded fp16 GEMM (kai_mmqh.cuh)
// A launch whose last round of workgroups would be a small fraction of the CUs: the tiles of a
// rectangle at the output's end (activation rows [r0, r0 + rows) = [r0, m), weight rows
// [c0, c0 + cols) = [c0, n), r0 and c0 on tile bounds) run in `splits` K pieces of `stages`
// stages whose fp32 sums go to scratch [piece][rows][cols] for mmqh_reduce_kernel; the other
// `main` tiles run whole (K unsplit). No tail: main is every tile and rows is 0.
struct MmqhTail {
    int main, splits, stages, r0, rows, c0, cols;
};
// The fp32 sums a call's scratch holds for an (n, k, m) product (kai_fused_mmq_workspace): a size that
// callers query and keep, so it is a rule of its own and the launch plan below works inside it. In
// tiles of 128 weight rows by 96, 128 or 256 activation rows on 256 CUs: a K split (at most 8) where
// the tiles do not fill the chip, or the K pieces (at most 8, at most 32 MiB) of the tiles that a
// last, at most half full round would hold, whichever a simple cost model prefers.
constexpr size_t MMQH_TAIL_BYTES = size_t(32) << 20;
constexpr int MMQH_CUS = 256;
inline size_t mmqh_sums_bytes(int type, int64_t n, int64_t k, int64_t m) {
    const int64_t bm = m <= 96 ? 96 : m > 128 && type != Q8_0 ? 256 : 128, bn = 128;
    const int64_t tn = (n + bn - 1) / bn, tm = (m + bm - 1) / bm, tiles = tn * tm;
    const int stages = static_cast<int>((k + 255) / 256 * 4);
    const double tile = double(bn / 32) * double(bm / 32), per_sum = 1.0 / (320.0 * double(k));
    double best = 1e300;
    int best_splits = 1;
    for (int want = 1; want <= 8; ++want) {
        const int chunk = ((stages + want - 1) / want + 3) / 4 * 4, splits = (stages + chunk - 1) / chunk;
        if (splits != want || (splits > 1 && chunk < 16)) continue;
        const double t = double((tiles * splits + MMQH_CUS - 1) / MMQH_CUS) * tile / splits +
                         (splits > 1 ? double(splits) * double(m) * double(n) * per_sum : 0.0);
        if (t < best) best = t, best_splits = splits;
    }
    const size_t split_bytes = best_splits > 1 ? size_t(best_splits) * size_t(m) * size_t(n) * sizeof(float) : 0;
    const int64_t rem = tiles % MMQH_CUS, full = tiles - rem;
    if (full == 0 || rem == 0 || 2 * rem > MMQH_CUS) return split_bytes;
    int64_t height = 1;  // the fewest activation tiles whose last weight tiles make `rem`
    while (height <= tm && (rem % height || rem / height > tn)) ++height;
    if (height > tm) return split_bytes;
    const int64_t rows = m - (tm - height) * bm, cols = n - (tn - rem / height) * bn;
    int64_t pieces = std::min<int64_t>({MMQH_CUS / rem, 8, stages / 4,
                                        static_cast<int64_t>(MMQH_TAIL_BYTES / size_t(rows * cols * 4))});
    if (pieces < 2) return split_bytes;
    const int chunk = static_cast<int>(((stages + pieces - 1) / pieces + 3) / 4 * 4);
    pieces = (stages + chunk - 1) / chunk;
    if (pieces < 2) return split_bytes;
    const double t = double(full / MMQH_CUS) * tile + tile * chunk / stages +
                     double(pieces) * double(rows) * double(cols) * per_sum;
    return t < best ? size_t(pieces) * size_t(rows) * size_t(cols) * sizeof(float) : split_bytes;
}

// Configurations: the whole-chip tile (256 x 256, 8 waves, one workgroup per CU); the general one
// (128 x 128, 4 waves, two per CU: its fine grid fills a last round, and one workgroup's waits
// overlap the other's work); between them 256 x 128 (8 waves), and 128 x 128 with K dealt to two
// groups of waves, for grids of fewer workgroups than CUs; for few rows 128 weight rows by 32, 64 or
// 96 activation rows with K dealt to GK groups of waves in the workgroup, which add their sums in LDS
// (so few rows leave one group's waves mostly waiting for their weights); and the same with 32
// weight rows, so that a matrix of a few thousand rows fills the chip too.
enum MmqhId : int {
    MMQH_WIDE, MMQH_TALL, MMQH_HALF, MMQH_HALF2, MMQH_ROWS32, MMQH_ROWS64, MMQH_ROWS96, MMQH_THIN32, MMQH_THIN64,
    MMQH_THIN96, MMQH_IDS
};
struct MmqhConfig {
    int bn, bm, slots;        // tile, resident workgroups of the chip
    double fixed, low, high;  // us of a workgroup: start and end, and a stage on an empty and a full chip
};
// Times measured on MI355X (16384 and 32768 x 4096 at 32 to 512 rows, half a chip and a whole one; Q8_0's
// and Q2_K's adjusted to calls of 70 shapes each on every configuration). The plan's choice was within 1-2 %
// of the best configuration's time on average over those shapes of every format.
inline MmqhConfig mmqh_config(MmqhId id, int type) {
    constexpr int TILE[MMQH_IDS][3] = {{256, 256, 256}, {256, 128, 256}, {128, 128, 512}, {128, 128, 256}, {128, 32, 256},
                                       {128, 64, 256},  {128, 96, 256},  {32, 32, 256},   {32, 64, 256},   {32, 96, 256}};
    constexpr double FIXED[MMQH_IDS] = {12.0, 8.0, 6.0, 6.0, 6.0, 6.0, 6.0, 4.5, 5.0, 5.0};
    constexpr double US[5][MMQH_IDS][2] = {
        // Q4_K
        {{1.30, 1.85}, {0.70, 1.13}, {0.45, 1.22}, {0.36, 0.63}, {0.26, 0.39}, {0.31, 0.50}, {0.36, 0.56}, {0.09, 0.13},
         {0.11, 0.16}, {0.18, 0.23}},
        // IQ3_S
        {{1.65, 2.10}, {1.20, 1.45}, {0.78, 1.50}, {0.60, 0.77}, {0.50, 0.58}, {0.52, 0.60}, {0.58, 0.68}, {0.15, 0.17},
         {0.19, 0.22}, {0.26, 0.29}},
        // Q4_0
        {{1.62, 2.10}, {1.00, 1.40}, {0.70, 1.45}, {0.45, 0.75}, {0.30, 0.45}, {0.35, 0.50}, {0.38, 0.57}, {0.14, 0.17},
         {0.18, 0.22}, {0.23, 0.27}},
        // Q8_0
        {{2.15, 2.36}, {1.43, 1.70}, {0.95, 1.83}, {0.60, 0.85}, {0.42, 0.62}, {0.46, 0.65}, {0.60, 0.73}, {0.18, 0.22},
         {0.25, 0.27}, {0.29, 0.33}},
        // Q2_K
        {{1.62, 2.04}, {0.70, 1.02}, {0.36, 1.10}, {0.36, 0.63}, {0.16, 0.31}, {0.22, 0.35}, {0.29, 0.45}, {0.10, 0.13},
         {0.15, 0.18}, {0.20, 0.28}}};
    const int f = type == IQ3_S ? 1 : type == Q4_0 ? 2 : type == Q8_0 ? 3 : type == Q2_K ? 4 : 0;
    return {TILE[id][0], TILE[id][1], TILE[id][2], FIXED[id], US[f][id][0], US[f][id][1]};
}
constexpr double MMQH_LAUNCH_US = 4.0, MMQH_SUMS_BYTES_PER_US = 4.5e6;

// Launch plan of an m-row product. It depends only on the type and shape (sized for the 256
// CUs of an MI355X).
struct MmqhPlan {
    MmqhId id = MMQH_HALF;
    int tiles_n = 0, tiles_m = 0, splits = 1, split_stages = 0;
    MmqhTail tail = {};
    int rest = 0;  // tiles left to a second launch, in MMQH_HALF's quarters
    double us = 1e300;
    bool has_tail() const { return tail.rows > 0; }
};
// A round's stage time between `low` and `high` by how much of the chip it uses; with two workgroups
// on some CUs those set the round's end.
inline double mmqh_rounds_us(const MmqhConfig &c, int64_t wgs, int stages) {
    const int64_t rem = wgs % c.slots;
    if (rem == 0) return double(wgs / c.slots) * (c.fixed + stages * c.high);
    const double f = double(rem) / MMQH_CUS, one = c.slots > MMQH_CUS ? 0.27 : 1.0;
    const double share = f <= 1.0 ? one * f * f : 0.7 + 0.3 * (f - 1.0);
    return double(wgs / c.slots) * (c.fixed + stages * c.high) + c.fixed + stages * (c.low + (c.high - c.low) * share);
}
inline void mmqh_consider(MmqhPlan &best, MmqhId id, int type, int64_t n, int64_t k, int64_t m, size_t sums) {
    const MmqhConfig c = mmqh_config(id, type);
    const int stages = static_cast<int>((k + 255) / 256 * 4);
    const int64_t tn = (n + c.bn - 1) / c.bn, tm = (m + c.bm - 1) / c.bm, tiles = tn * tm;
    auto take = [&](double us, int splits, int chunk, const MmqhTail &tail, int rest) {
        if (us >= best.us) return;
        best = {id, static_cast<int>(tn), static_cast<int>(tm), splits, chunk, tail, rest, us};
    };
    const MmqhTail none = {static_cast<int>(tiles), 1, 0, 0, 0, 0, 0};
    for (int want = 1; want <= 8; ++want) {
        const int chunk = ((stages + want - 1) / want + 3) / 4 * 4, splits = (stages + chunk - 1) / chunk;
        const double bytes = double(splits) * double(m) * double(n) * 4;
        if (splits != want || (splits > 1 && (chunk < 8 || bytes > double(sums)))) continue;
        take(mmqh_rounds_us(c, tiles * splits, chunk) +
                 (splits > 1 ? MMQH_LAUNCH_US + 2 * bytes / MMQH_SUMS_BYTES_PER_US : 0.0),
             splits, chunk, none, 0);
    }
    const int64_t rem = tiles % c.slots, full = tiles - rem;
    if (full == 0 || rem == 0) return;
    if (id == MMQH_WIDE) {  // the last round's tiles in quarters
        MmqhTail whole = none;
        whole.main = static_cast<int>(full);
        take(mmqh_rounds_us(c, full, stages) + mmqh_rounds_us(mmqh_config(MMQH_HALF, type), 4 * rem, stages) + MMQH_LAUNCH_US / 2,
             1, stages, whole, static_cast<int>(rem));
    }
    // the last round's tiles, as a rectangle of the fewest activation tiles, in K pieces
    int64_t height = 1;
    while (height <= tm && (rem % height || rem / height > tn)) ++height;
    if (height > tm) return;
    const int64_t r0 = (tm - height) * c.bm, c0 = (tn - rem / height) * c.bn, rows = m - r0, cols = n - c0;
    int64_t pieces = std::min<int64_t>({c.slots / rem, 8, stages / 4, static_cast<int64_t>(sums / size_t(rows * cols * 4))});
    if (pieces < 2) return;
    const int chunk = static_cast<int>(((stages + pieces - 1) / pieces + 3) / 4 * 4);
    pieces = (stages + chunk - 1) / chunk;
    if (pieces < 2) return;
    take(mmqh_rounds_us(c, full, stages) + mmqh_rounds_us(c, rem * pieces, chunk) + MMQH_LAUNCH_US +
             8.0 * double(pieces) * double(rows) * double(cols) / MMQH_SUMS_BYTES_PER_US,
         1, stages,
         {static_cast<int>(full), static_cast<int>(pieces), chunk, static_cast<int>(r0), static_cast<int>(rows),
          static_cast<int>(c0), static_cast<int>(cols)},
         0);
}
// Every configuration is considered at every number of rows: a rule that kept the 32-, 64- and 96-row
// tiles to at most 192 rows left narrow and mid-sized products on tiles twice their need (us, whole
// calls: Q8_0 512 x 5120 at 97 rows 26.1 -> 17.9, 140 x 1216 at 312 rows 26.8 -> 15.8; Q4_0
// 9892 x 5792 at 242 rows 74.6 -> 58.2).
inline MmqhPlan mmqh_plan(int type, int64_t n, int64_t k, int64_t m) {
    MmqhPlan best;
    const size_t sums = mmqh_sums_bytes(type, n, k, m);
    for (int id = 0; id < MMQH_IDS; ++id) mmqh_consider(best, MmqhId(id), type, n, k, m, sums);
    return best;
}

// ------------------------------------------------------------------------------ Q6_K (kai_mmq6.cuh)
// Tile configurations of the Q6_K batched GEMM (kai_mmq6.cuh): activation rows, weight rows, K groups (four waves two workgroups to a CU,
// else eight waves to a CU).
enum Mmq6Id : int { MMQ6_NONE = -1, MMQ6_96X128, MMQ6_96X128_2, MMQ6_96X64_4, MMQ6_64X64_4, MMQ6_IDS };
// Which one an m-row product of an n x k matrix takes, or MMQ6_NONE: the int8 tile kernel
// (kai_mmq.cuh), whose many small tiles are faster up to 80 rows and on matrices of few rows. Its
// time is taken as the padded work at 184 TOP/s. Measured on MI355X (kernel alone, us; stage times
// below from the same runs): 5120 x 17408 at 96 / 160 / 256 / 512 rows int8 tiles 114 / 232 / 262 / 412,
// here 129 / 133 / 176 / 281; 5120 x 6144 at 96 / 160 rows 42 / 84, here 52 / 55; 34816 x 5120 at 64 / 96
// rows 134 / 251, here 154 / 163; 512 x 5120 at 160 / 1000 rows 15 / 40, here 39 / 41.
inline Mmq6Id mmq6_plan(int64_t n, int64_t k, int64_t m) {
    struct Config {
        int bm, bn, slots;
        double low, high;  // us of a stage, up to one workgroup per CU and with two
    };
    constexpr Config CONFIGS[MMQ6_IDS] = {{96, 128, 512, 1.22, 1.80}, {96, 128, 256, 1.03, 1.16}, {96, 64, 256, 0.60, 0.65},
                                          {64, 64, 256, 0.48, 0.50}};
    if (m <= 80) return MMQ6_NONE;
    const double stages = double(k) / 64, padded = double((m + 63) / 64 * 64);
    double best = 2.0 * padded * double(n) * double(k) / 184e6;
    Mmq6Id id = MMQ6_NONE;
    for (int c = 0; c < MMQ6_IDS; ++c) {
        const Config &f = CONFIGS[c];
        const int64_t wgs = (n + f.bn - 1) / f.bn * ((m + f.bm - 1) / f.bm), rem = wgs % f.slots;
        const double us = double(wgs / f.slots) * (6.0 + stages * f.high) +
                          (rem ? 6.0 + stages * (rem <= 256 && f.slots > 256 ? f.low : f.high) : 0.0);
        if (us < best) best = us, id = Mmq6Id(c);
    }
    return id;
}
}  // namespace kai
