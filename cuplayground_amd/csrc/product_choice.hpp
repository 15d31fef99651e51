// Whether a 16-bit weight gradient takes its operands as they are stored (the 128 x 128 tiles of ffn_bf16_grouped.hip that turn them round on
// the way) or transposed copies of them and the larger tiles, and which tile a data gradient takes.  Either way gives the same bits.  Host arithmetic only, so that a host
// program can test it.  Estimates of either, us; constants and checks are measurements of whole calls (transposes and launches included,
// bf16, one card):
//   hand-ordered 256 x 256 tile: 1.3 us a slab of 64 and 8 us a task, rounds of 256 tasks and half a one; transposes at 4.5 TB/s read and
//   written;  as stored: 1.25 us a slab and round of 512 tasks (two on a compute unit share its time), 5 us a round.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstdint>

#include "two_launches.hpp"

namespace moe355 {

// The hand-ordered slab loop needs 32-bit buffer offsets: operands below 4 GiB, and for the weights also the columns behind the last one
// that a ragged tile reaches.  Dimensions are multiples of 64 (moe_config_validate).
constexpr int64_t kBufferLimit = (int64_t)1 << 32;
inline bool hand_weights_ok(int64_t N, int64_t K) { return (N + 256) * K * 2 < kBufferLimit; }
inline int columns256(int N) { return (N + 255) / 256; }

// Transposed operands of a weight gradient: an expert's window of columns is padded to kWindowAlign, rows are wgrad_ld long.
constexpr int kWindowAlign = 128;
inline int64_t wgrad_ld(int64_t A, int E) { return (A + (int64_t)kWindowAlign * E + 127) / 128 * 128; }
// They take the hand-ordered tile, else the 128 x 128 tile of the general loop.
inline bool wgrad_hand_ok(int N, int K, int64_t ld) { return N >= 1024 && K >= 1024 && hand_weights_ok(N, ld) && hand_weights_ok(K, ld); }

inline double stored_us(double tiles, double slabs) { return std::max(tiles / 512, 1.0) * (1.25 * slabs + 5.0); }
inline double transposed_us(double tiles, double slabs, double transposed_bytes) {
    const double rounds = tiles / 256;
    return (rounds <= 1.0 ? 1.0 : rounds + 0.5) * (1.3 * slabs + 8.0) + 2.0 * transposed_bytes / 4.5e6 + 8.0;
}
inline bool stored_operands_ok(int64_t rows, int N, int K) {
    return (rows + 128) * std::max(N, K) * 2 < kBufferLimit && (int64_t)(N + 128) * K * 2 < kBufferLimit && (int64_t)(K + 128) * N * 2 < kBufferLimit;
}

// Weight gradient [E, N, K] of A rows.  Transposed / as stored: 16 experts of 2048 x 2048, 512 rows each 124 / 105; 750 rows of 1408 x 2048
// 127 / 98; 136 of 1280 x 1408 48 / 27; 19 of 1024 x 2560 48 / 22; 4 of 2048 x 2560, 4096 rows 231 / 201; 64 of 1408 x 2048, 1536 rows
// 856 / 717; 16 of 2048 x 2560, 1024 rows 230 / 224 (estimated the other way round); 8 of 4096 x 2048, 2048 rows 305 / 330; 8 of 4096 x
// 14336, 512 rows 641 / 721, 2048 rows 1710 / 2229.  Behind the general loop: 8 of 960 x 14336, 4096 rows 1494 / 1105; 64 of 960 x
// 4096, 2048 rows 1945 / 1319; 12 of 512 x 512, 100 rows 18.5 / 9.1 (16 shapes in bf16 and fp16: as stored takes 0.44 to 0.77 of the time).
inline bool wgrad_as_stored(int64_t A, int E, int N, int K) {
    if (!stored_operands_ok(A, N, K)) return false;
    if (!wgrad_hand_ok(N, K, wgrad_ld(A, E))) return true;
    const double rows = (double)A / std::max(E, 1);
    return stored_us((double)E * ((N + 127) / 128) * ((K + 127) / 128), rows / 64 + 0.5) <
           transposed_us((double)E * columns256(N) * columns256(K), rows / 64 + 1.0, 2.0 * A * (N + K));
}
// As stored on the 256 x 256 tile whose workgroups stay (wgrad_ring_kernel): where the 128 x 128 tiles lose to transposed copies, and
// where it beats them by whole rounds, us: 8.5 a task of 256 and 1.3 a slab (an odd number of slabs is one more), against 3.6 and 1.1 a
// round of 512.  This / 128 x 128 tiles: 16 experts of 2048 x 2048, 512 rows each 81 / 101; of 2048 x 1408, 750 rows 82 / 96; 4 of 2048 x
// 2560, 4096 rows 174 / 192; 4 of 1024 x 2560, 750 rows 27 / 31; 8 of 1920 x 1536, 500 rows 41 / 43; 8 of 1024 x 2560, 750 rows 50 / 50; 8 of
// 1280 x 1664, 250 rows 29 / 27; 16 of 1152 x 1920, 175 rows 44 / 36; 16 of 1024 x 2560, 19 rows 32 / 23.
inline bool wgrad_large(int64_t A, int E, int N, int K, int products = 1) {      // (`products` of them, N x K or K x N, in one launch)
    if (!wgrad_as_stored(A, E, N, K)) return true;
    const double slabs = (double)A / std::max(E, 1) / 64, experts = (double)products * E;
    const double large = std::ceil(experts * columns256(N) * columns256(K) / 256) * (1.3 * (slabs + 1.0) + 8.5);
    const double small = std::ceil(experts * ((N + 127) / 128) * ((K + 127) / 128) / 512) * (1.1 * (slabs + 0.5) + 3.6);
    return large < small;
}
// Data gradient [A, N] from rows of K and the weight [E, K, N]: as stored wherever the offsets allow it -- the transposing fragment reads
// (ffn_bf16_tile.hpp) run at the rate of the plain ones, and the transposed copy costs what it moves.
inline bool grouped_kn_as_stored(int64_t A, int, int N, int K) { return stored_operands_ok(A, N, K); }
// ... on 256-row blocks and remainders, or on 128-row blocks: the shorter by the estimate of a layer's launches (two_launches.hpp).
// us, 256 / 128: 16 experts of 2048 x 2048, 512 rows each 81 / 86; of 1408 x 2048, 750 rows 77 / 90; 4 of 2560 x 2048, 4096 rows 133 / 157; 8 of
// 1664 x 1280, 250 rows 40 / 25; 16 of 1920 x 1152, 175 rows 45 / 28; 8 of 2560 x 1024, 750 rows 59 / 40; 4 of them 55 / 34; 8 of 1536 x
// 1920, 500 rows 41 / 46 (the 128 x 128 tiles that turned the operand round in registers: 107, 107, 230, 27, 41, 56, 37, 38).
inline bool grouped_kn_large(int64_t A, int E, int N, int K, int products = 1) {      // (`products` of this shape in one launch)
    const SplitBlocks n(A, std::max(E, 1));
    const double cols = products * columns256(N);
    return split_us(n.full * cols, n.left * cols, K) < split_us(0, n.small * cols, K);
}

}  // namespace moe355
