// Which tile of a grouped product (packed rows, a matrix per expert) a workgroup takes, from the experts' row counts alone.
#pragma once

#include "ffn_common.hpp"

namespace moe355 {
namespace {

constexpr int kShareSlack = 14;      // workgroups without a tile, at most: the two lists are rounded up to eight equal shares
// Row blocks of an expert that are taken at a time, all column tiles of those: the 32 tiles that an XCD works on then share 8 row
// blocks and 4 weight tiles instead of one weight tile.  One expert's row blocks all at a time / 8, us: one expert of 4096 x 4096, 8192
// rows, up projection 220 / 208, its data gradient 236 / 225; 2 of them 251 / 246; 8 of 1408 x 2048, 4096 rows 201 / 197; 4 of 2048 x 2048,
// 3072 rows 113 / 109; 4 of 2560 x 2048, 4096 rows 144 / 146; a layer of one expert of 2048 x 2048, SwiGLU, 8192 rows 218 / 212.
constexpr int kRowChunk = 8;
struct GroupedTask {
    int expert, row0, rows, ctile;
};
// Which tile workgroup `id` of a grouped product takes, from the experts' row counts alone; false: none.  Order: the row blocks of
// full height, expert by expert, column tile by column tile, an expert's row blocks (kRowChunk of them) fastest (few row blocks stay in the
// caches while its column tiles pass by); with 256-row blocks, behind them the remainders of at most 128 rows: the long tasks start
// first, and the short ones fill the compute units that the last round of long ones leaves idle.  Workgroups go to the eight XCDs in
// turn: each XCD takes an eighth of either list in a row, so that the tiles that share a weight tile or token rows share an L2.
// Every wavefront works it out for itself, an expert a lane, which takes less time than a launch in front that writes tables.
// One product, bf16, the launch and table in front of 256-row blocks alone against this: 16 experts of 2048 x 2048, about 512 rows each
// 109 -> 80 us; 8 of 4096 x 2048, 2048 rows 274 -> 234; 64 of 2048 x 1408, 94 rows 94 -> 89; 16 of 2048 x 1408, 750 rows 91 -> 73.
// The share of an XCD in a row, against the list dealt out to them: whole layers as two launches, 8 experts of 4096 x 14336, 2048 rows
// 4679 -> 4431 us, 1024 rows 2860 -> 2484; 64 of 2048 x 1408, 1536 rows 1863 -> 1662, 750 rows 1089 -> 907; 12 of 1344 x 2752, 444 rows
// 174 -> 165, 150 rows 125 -> 107.
template <int BIG>
__device__ __forceinline__ bool grouped_task(const int32_t* __restrict__ count, const int32_t* __restrict__ offset, int E, int ncol, int id, GroupedTask& t) {
    constexpr int LEFT = BIG == 256 ? 128 : 0;          // rows up to which what is left of an expert is a block of its own kind
    const int lane = threadIdx.x & 63;
    auto rows_of = [&](int c) { return c + lane < E ? max(count[c + lane], 0) : 0; };
    auto big_of = [&](int n) { return (n + BIG - 1 - LEFT) / BIG; };
    int big_sum = 0, left_sum = 0;         // full row blocks and remainders of all experts
    for (int c = 0; c < E; c += kWave) {
        const int n = rows_of(c), big = big_of(n);
        big_sum += big;
        left_sum += n > big * BIG ? 1 : 0;
    }
#pragma unroll
    for (int off = kWave / 2; off; off >>= 1) {
        big_sum += __shfl_xor(big_sum, off, kWave);
        left_sum += __shfl_xor(left_sum, off, kWave);
    }
    const int bigs = __builtin_amdgcn_readfirstlane(big_sum) * ncol, lefts = __builtin_amdgcn_readfirstlane(left_sum) * ncol;
    const int big_share = (bigs + 7) / 8, left_share = (lefts + 7) / 8;
    if (id < 8 * big_share) {
        id = (id & 7) * big_share + (id >> 3);
        if (id >= bigs) return false;
    } else {
        id -= 8 * big_share;
        if ((id >> 3) >= left_share) return false;
        id = (id & 7) * left_share + (id >> 3) + bigs;
        if (id >= bigs + lefts) return false;
    }
    int base = 0;                          // full row blocks of the experts in front
    for (int c = 0; c < E; c += kWave) {
        const int n = rows_of(c), big = big_of(n);
        int inc = big;
#pragma unroll
        for (int off = 1; off < kWave; off <<= 1) {
            const int o = __shfl_up(inc, off, kWave);
            if (lane >= off) inc += o;
        }
        const int total = __builtin_amdgcn_readlane(inc, kWave - 1);
        if (id < (base + total) * ncol) {
            const int l = __builtin_ctzll(__ballot((base + inc) * ncol > id));
            const int blocks = __builtin_amdgcn_readlane(big, l), first = base + __builtin_amdgcn_readlane(inc, l) - blocks;
            int local = id - first * ncol, rb = 0, width = blocks;
            if (blocks > kRowChunk) {
                rb = local / (kRowChunk * ncol) * kRowChunk;
                width = min(kRowChunk, blocks - rb);
                local -= rb * ncol;
            }
            t.ctile = local / width;
            rb += local - t.ctile * width;
            t.expert = c + l;
            t.rows = min(BIG, __builtin_amdgcn_readlane(n, l) - rb * BIG);
            t.row0 = offset[t.expert] + rb * BIG;
            return true;
        }
        base += total;
    }
    if constexpr (LEFT > 0) {
        int before = (id - base * ncol) / ncol;      // remainders in front of this one
        t.ctile = (id - base * ncol) - before * ncol;
        for (int c = 0; c < E; c += kWave) {
            const int n = rows_of(c), left = max(n - big_of(n) * BIG, 0);
            const unsigned long long m = __ballot(left > 0);
            const int here = __popcll(m);
            if (before < here) {
                const int rank = __popcll(m & ((1ull << lane) - 1ull));
                const int l = __builtin_ctzll(__ballot(((m >> lane) & 1) && rank == before));
                t.expert = c + l;
                t.rows = __builtin_amdgcn_readlane(left, l);
                t.row0 = offset[t.expert] + (__builtin_amdgcn_readlane(n, l) - t.rows);
                return true;
            }
            before -= here;
        }
    }
    return false;
}

}  // namespace
}  // namespace moe355
