// Which 16-bit layers on the hand-ordered tiles run as two launches (ffn_bf16_grouped.hip: launch_ffn_split_16) instead of on the task
// queue, and on which row blocks.  Host arithmetic on the layer's shape only, so that a host program can test it.  "Queue / two" below
// are whole layers, us, bf16, tokens from one seed, both modes of one handle's shape in turn on one card; "random layers" are 300 with
// 4 to 64 experts, 60 to 500 rows each and dimensions of 512 to 4096 in steps of 64.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstdint>

namespace moe355 {

// Time of one task of a grouped product, us, from its contraction's length: 256 x 256 (large) or 128 x 256 tile; cold weights; the fill of
// the first slabs, epilogue and launch or queue overhead in the constant.
inline double tile_task_us(bool large, int K) {
    const double slabs = (K + 63) / 64;
    return large ? 1.3 * slabs + 10.0 : 1.1 * slabs + 3.0;
}

struct TwoLaunchShape {
    int64_t pairs;               // packed rows at most: tokens x experts per token
    int experts, H, I;
    bool swiglu;
    int columns_up() const { return (I * (swiglu ? 2 : 1) + 255) / 256; }
    int columns_down() const { return (H + 255) / 256; }
};

constexpr int kTaskUnits = 256;  // compute units: one task each at a time

// AUTO on 128-row blocks (large = false): always, unless tokens are dropped and an expert takes at most kSplitCappedRows.
//   Random layers: two launches are faster at 176 of 179, by a fifth in the mean.  The others: 32 of 2944 x 2688, GELU, 71 rows 8 % slower, 64
//   of 2432 x 1664, SwiGLU, 101 rows 5 %, 9 of 2048 x 2112, SwiGLU, 388 rows (on 128-row blocks; it runs on 256-row ones).
//   Dropping layers, 64 of 2048 x 1408: at most 29 rows 234 / 243, 38 rows 237 / 247, 57 rows 248 / 248, 94 rows 249 / 240 (28 rows, none
//   dropped: 284 / 267).
// On 256-row blocks the queue starts the down projection under the up projection's last round, which two launches have to make up for:
//   few rows an expert, where remainders are most of the work and a remainder's task is shorter here: 64 of 2048 x 1408, 137 to 188 rows
//   3 to 6 % faster, 197 rows of 32 of 3456 x 3264 6 % slower; at most 192 rows, random layers: faster at 25 of 26 (64 of 3072 x 1600, 125
//   rows, 3 % slower; another, 32 of 3392 x 2560, ReLU, 166 rows, 8 %: 1.25 and 1.75 rounds, which two launches make two and two);
//   many rounds of tasks whose rows stay in the caches: the queue's pops and written-through rows add up, but each XCD works on an expert
//   of its own, so that the rows of eight experts are read at a time, where the queue's workgroups share one expert's.  Bytes of eight
//   experts' rows, 11 to 16 rounds, none dropped, queue / two:
//     up to 78 MB: 64 of 2048 x 1408, 1434 rows 1606 / 1574, 1792 rows 1985 / 1935; 64 of 4096 x 1536, 956 rows 2239 / 2208; 64 of
//     1536 x 1536, 1911 rows 1404 / 1363; 128 of 1024 x 1024, 1434 rows 1298 / 1264; routed like 1 / rank^0.5 and 1 / rank^1.1 0.5 % slower to
//     16 % faster;
//     94 to 161 MB: 32 of 2048 x 2048, 2867 rows 1646 / 1623 but like 1 / rank^1.1 1679 / 1724; 32 of 2048 x 2816, 3584 rows 3467 / 3426, 3477 / 3642;
//     134 to 1600 MB: 16 of 3072 x 3072, 2731 rows 1542 / 1567; 8 of 4096 x 4096, 5734 rows 3607 / 3824; 8 of 4096 x 14336, 5734 rows
//     12213 / 12609, 7168 rows 15209 / 16273.
//   8 rounds of 64 of 2048 x 1408: 1167 / 1172.  Where tokens are dropped it depends on the routing, which is not known here (64 of
//   2048 x 1408, 1434 rows at most, even 1587 / 1542, like 1 / rank^1.1 704 / 714): the queue.
constexpr int kSplitRowsPerExpert = 192, kSplitRounds = 11, kSplitCappedRows = 48;
constexpr int64_t kSplitRowBytes = 80 << 20;
inline bool two_launches_auto(const TwoLaunchShape& s, bool large, bool drops, int64_t capacity) {
    if (!large) return !(drops && capacity <= kSplitCappedRows);
    if (s.pairs <= (int64_t)s.experts * kSplitRowsPerExpert) return true;
    const int64_t rounds = s.pairs / 256 * std::min(s.columns_up(), s.columns_down()) / kTaskUnits;
    const int64_t row_bytes = 8 * (s.pairs / s.experts) * std::max(s.H, s.I) * 2;
    return rounds >= kSplitRounds && !drops && row_bytes <= kSplitRowBytes;
}

// Time of a launch of `full` tasks of `large` each and, behind them, `left` tasks of `small`.
inline double split_time(double full, double left, double large, double small) {
    const double whole = std::floor(full / kTaskUnits), busy = full - whole * kTaskUnits, idle = kTaskUnits - busy;
    double at_idle = whole * large, at_busy = (whole + 1) * large, end = busy > 0 ? at_busy : at_idle;
    while (left > 0) {
        const bool first = busy <= 0 || at_idle <= at_busy;
        double& at = first ? at_idle : at_busy;
        left -= first ? idle : busy;
        at += small;
        end = std::max(end, at);
    }
    return end;
}
inline double split_us(double full, double left, int K) { return split_time(full, left, tile_task_us(true, K), tile_task_us(false, K)); }
// Of `pairs / experts` rows per expert on average, an expert has about that +- its root: tiles per column tile of all experts.
struct SplitBlocks {
    double full = 0, left = 0, small = 0, table = 0;      // 256-row blocks and remainders; or 128-row blocks; or 256-row blocks alone
    SplitBlocks(int64_t pairs, int experts) {
        const double rows = (double)pairs / experts;
        for (int i = -1; i <= 1; ++i) {
            const double n = std::max(1.0, std::round(rows + i * std::sqrt(rows))), share = experts * (i ? 0.25 : 0.5), f = std::floor((n + 127) / 256);
            full += share * f;
            left += n > 256 * f ? share : 0;
            small += share * std::ceil(n / 128);
            table += share * std::ceil(n / 256);
        }
    }
};
// Layers planned on 128-row blocks whose two launches take 256-row blocks and remainders after all: where a second block of an expert, or a
// round of them, would be opened for a few rows.  128-row blocks / these: 18 of 1856 x 2944, SwiGLU, 157 rows 277 / 205; 17 of 2048 x 2048,
// ReLU, 156 rows 187 / 138; 24 of 1536 x 1600, ReLU, 148 rows 131 / 109; 64 of 960 x 896, GELU, 212 rows 13 % faster.  The estimate has to
// promise a tenth: of 219 layers planned on 128-row blocks it moves 29, 23 of them 6 to 26 % faster, 6 of them 1 to 10 % slower; of another
// 110 that it moves 89 are up to 28 % faster, 21 are 1 to 13 % slower (9 of 1216 x 2688, ReLU, 649 rows).  With a 128-row tile at three
// quarters of a round whatever the contraction's length it moves 43 of the 219, 19 of them up to 24 % slower (23 of 768 x 704, 143 rows 64 / 80).
inline bool two_launches_on_256(const TwoLaunchShape& s) {
    const SplitBlocks n(s.pairs, s.experts);
    const double up = s.columns_up(), down = s.columns_down();
    const double large = split_us(n.full * up, n.left * up, s.H) + split_us(n.full * down, n.left * down, s.I);
    const double small = split_us(0, n.small * up, s.H) + split_us(0, n.small * down, s.I);
    return large <= 0.9 * small;
}
// Layers of 8 or 16 experts on 256-row blocks whose full row blocks are a round of their own in the up projection, so that the remainders'
// round reads all weights from memory again, and that take as many rounds on 256-row blocks alone: the order of the row block table,
// where the blocks of an expert meet the same weight tile, is kept.  Table / remainders behind: 16 of 2048 x 2048, SwiGLU, 260 rows 187 / 193,
// 278 rows 186 / 218, 300 rows 188 / 233, 325 rows 189 / 235; but 237 rows 202 / 181 (hardly a remainder), GELU (one round) 325 rows 155 / 144.
// 16 of 3904 x 1856, SwiGLU, 306 rows: the up projection fetches 0.95 GB with remainders behind, 0.50 in the table's order.  Of 16 random
// layers of 8 or 16 experts with full blocks of 0.9 rounds and more 14 are up to 15 % faster, 2 are 0.2 and 3 % slower; of 11 with 0.8 to
// 0.9 rounds of 32 slabs and more 10 are 4 to 13 % faster, one is 4 % slower, and 3 of fewer slabs are 2 to 9 % slower.  With other numbers of experts (an XCD's
// share of the list then begins and ends inside an expert, and the table's columns are dealt out unevenly) remainders behind are faster at 27
// of 30, by up to 30 %: 24 of 1600 x 2112, GELU, 370 rows fetch 0.31 GB against 0.39; 22 of 1216 x 2752, GELU, 309 rows 272 / 184; 24 of 1024 x
// 2560, 303 rows 43 % more on the table; the other way round 10 of 1920 x 2944, SwiGLU, 373 rows 188 / 198, 12 of 3712 x 3904, 17 of 3456 x
// 3776 and 29 of 1920 x 1984 2 to 3 %.
inline bool two_launches_keep_table(const TwoLaunchShape& s) {
    const SplitBlocks n(s.pairs, s.experts);
    const double up = s.columns_up(), down = s.columns_down();
    auto rounds = [](double tiles) { return std::ceil(tiles / kTaskUnits); };
    return s.experts % 8 == 0 && s.experts <= 16 && n.left >= 0.75 * s.experts && n.full <= 1.25 * s.experts && n.full * up >= (s.H >= 2048 ? 0.8 : 0.9) * kTaskUnits && rounds(n.table * up) <= 2 &&
           rounds(n.table * down) <= std::ceil(split_time(n.full * down, n.left * down, 1.0, 0.75) - 0.5);      // (in rounds: a remainder is 0.74 at 32 slabs)
}

}  // namespace moe355
