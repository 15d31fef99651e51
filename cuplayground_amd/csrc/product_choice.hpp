// Which tiles the 16-bit products of a training step take: a weight gradient's (ffn_bf16_grouped.hip: wgrad_rows_kernel on 128 x 128 tiles,
// wgrad_ring_kernel on 256 x 256) and a data gradient's.  Both read their operands as they are stored, and either choice gives the same
// bits.  Host arithmetic only, so that a host program can test it.
#pragma once
#include <algorithm>
#include <cstdint>

#include "two_launches.hpp"

namespace moe355 {

// The hand-ordered slab loop needs 32-bit buffer offsets: operands below 4 GiB, and for the weights also the columns behind the last one
// that a ragged tile reaches.  Dimensions are multiples of 64 (moe_config_validate).
constexpr int64_t kBufferLimit = (int64_t)1 << 32;
inline bool hand_weights_ok(int64_t N, int64_t K) { return (N + 256) * K * 2 < kBufferLimit; }
inline int columns256(int N) { return (N + 255) / 256; }
constexpr int kSlabRows = 64;        // of a weight gradient's sum, a step

// Where operands cannot be taken as stored (an option asks for a tile, pointers are unaligned, 4 GiB) a weight gradient works on
// transposed ones: an expert's window of columns is padded to kWindowAlign, rows are wgrad_ld long.
constexpr int kWindowAlign = 128;
inline int64_t wgrad_ld(int64_t A, int E) { return (A + (int64_t)kWindowAlign * E + 127) / 128 * 128; }
// They take the hand-ordered tile, else the 128 x 128 tile of the general loop.
inline bool wgrad_hand_ok(int N, int K, int64_t ld) { return N >= 1024 && K >= 1024 && hand_weights_ok(N, ld) && hand_weights_ok(K, ld); }

// Operands as stored wherever the offsets allow it: the transposing fragment reads (ffn_bf16_tile.hpp) run at the rate of the plain ones,
// and a transposed copy costs what it moves.
inline bool stored_operands_ok(int64_t rows, int N, int K) {
    return (rows + 128) * std::max(N, K) * 2 < kBufferLimit && (int64_t)(N + 128) * K * 2 < kBufferLimit && (int64_t)(K + 128) * N * 2 < kBufferLimit;
}

// A weight gradient [E, N, K] of A rows (`products` of them, N x K or K x N, in one launch) on the 256 x 256 tile, or on 128 x 128 ones.
// An expert's tiles are dealt out to the eight XCDs in equal shares, rounded up (WgradTiles::place), so that a launch takes as many rounds
// as the first XCD does, of 32 large tiles or 64 small ones: 64 experts of 384 x 256 have two large tiles each, on two XCDs.  A tile
// costs whole slabs of 64 rows, the large one an even number of them.  Large / small, us, one, two, three products:
//   16 experts of 2048 x 2048, 512 rows each 81 / 101 (one); 16 of 2048 x 2560, 1024 rows 161 / 230, 324 / 465, 480 / 684; 8 of 4096 x 4096, 300 rows 137 /
//   148, 274 / 339, 409 / 503; 8 of 4096 x 14336, 64 rows 269 / 268, 532 / 534, 793 / 798; 8 of 960 x 4096, 512 rows 46 / 56, 86 / 106, 124 / 166;
//   1 of 1024 x 4096, 8192 rows 152 / 98, 152 / 158, 169 / 238; 12 of 512 x 512, 2000 rows 47 / 30, 63 / 55, 116 / 87; 2 of 1536 x 1536, 8192 rows 151 / 145,
//   155 / 227, 202 / 311; 64 of 384 x 256, 112 rows 49 / 24 (two); 12 of 1408 x 640, 132 rows 29 / 16 (one).
// Of 11205 products of random sizes (1 to 64 experts, 256 to 3072 columns, 30 to 4000 rows; one to three of them) the estimate takes the
// slower tile by more than a tenth at 114, at most by 26 %.  Counting the tiles of all XCDs together, and taking the large tile wherever the
// small one was expected to lose to transposed copies: 552, up to twice the time.
inline bool wgrad_large(int64_t A, int E, int N, int K, int products = 1) {
    const int64_t experts = (int64_t)products * E, slab_rows = (int64_t)std::max(E, 1) * kSlabRows, slabs = (A + slab_rows - 1) / slab_rows;
    auto rounds = [&](int64_t tiles, int64_t per_xcd) { return (experts * ((tiles + 7) / 8) + per_xcd - 1) / per_xcd; };
    const double large = rounds((int64_t)columns256(N) * columns256(K), 32) * (1.2 * (slabs + slabs % 2) + 8.5);
    const double small = rounds((int64_t)((N + 127) / 128) * ((K + 127) / 128), 64) * (1.1 * slabs + 4.3);
    return large < small;
}

// A data gradient [A, N] from rows of K and the weight [E, K, N] on 256-row blocks and remainders, or on 128-row blocks: the shorter by
// the estimate of a layer's launches (two_launches.hpp; of 7470 random products, one or two in a launch, 188 by more than a tenth longer).
// us, 256 / 128: 16 experts of 2048 x 2048, 512 rows each 81 / 86; of 1408 x 2048, 750 rows 77 / 90; 4 of 2560 x 2048, 4096 rows 133 / 157; 8 of
// 1664 x 1280, 250 rows 40 / 25; 16 of 1920 x 1152, 175 rows 45 / 28; 8 of 2560 x 1024, 750 rows 59 / 40; 4 of them 55 / 34; 8 of 1536 x
// 1920, 500 rows 41 / 46 (the 128 x 128 tiles that turned the operand round in registers: 107, 107, 230, 27, 41, 56, 37, 38).
inline bool grouped_kn_large(int64_t A, int E, int N, int K, int products = 1) {      // (`products` of this shape in one launch)
    const SplitBlocks n(A, std::max(E, 1));
    const double cols = products * columns256(N);
    return split_us(n.full * cols, n.left * cols, K) < split_us(0, n.small * cols, K);
}

}  // namespace moe355
