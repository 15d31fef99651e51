// Which fp32 layers on the 128 x 128 matrix-core tile run on bf16 pieces instead (ffn_f32_pieces.hip), and on which row blocks.  Host
// arithmetic on the layer's shape only, so that a host program can test it.
#pragma once
#include "two_launches.hpp"

namespace moe355 {

struct PieceShape {
    int64_t tokens, pairs;
    int experts, H, I;
    bool swiglu;
    int64_t capacity;            // rows an expert keeps at most (pairs: none dropped)
    int columns_up() const { return (I * (swiglu ? 2 : 1) + 255) / 256; }
    int columns_down() const { return (H + 255) / 256; }
    // Dropping binds: nearly every expert is expected to keep `capacity` rows.
    bool capped() const { return (double)capacity * experts < 0.9 * pairs; }
};
// Row blocks of experts that have exactly `rows` rows each.
inline SplitBlocks exact_blocks(int64_t rows, int experts) {
    SplitBlocks n(rows, 1);
    n.full = (double)((rows + 127) / 256) * experts;
    n.left = rows > (rows + 127) / 256 * 256 ? experts : 0;
    n.small = (double)((rows + 127) / 128) * experts;
    return n;
}
inline SplitBlocks piece_blocks(int64_t pairs, int experts) { return experts == 1 ? exact_blocks(pairs, 1) : SplitBlocks(pairs, experts); }
// A projection's launch: 256-row blocks and remainders, or 128-row blocks; the shorter by the estimate of a layer's launches, the
// contraction six times as long.
inline bool pieces_large(int64_t pairs, int experts, int columns, int K) {
    const SplitBlocks n = piece_blocks(pairs, experts);
    return split_us(n.full * columns, n.left * columns, 6 * K) <= split_us(0, n.small * columns, 6 * K);
}

// The FFN stage on pieces, us.  10 bytes a value for the pieces of tokens and weights; a task's slab is the longer the more compute units
// are at work (the power limit): 0.7 to 1.3 us on the large tile, 0.35 to 1.1 on the small one.
inline double pieces_us(const PieceShape& s) {
    const SplitBlocks n = s.capped() ? exact_blocks(s.capacity, s.experts) : piece_blocks(s.pairs, s.experts);
    auto launch = [&](int columns, int K) {
        const double slabs = 6.0 * K / 64;
        const bool large = pieces_large(s.pairs, s.experts, columns, K);
        const double full = large ? n.full * columns : 0, left = (large ? n.left : n.small) * columns, fill = std::min(1.0, (full + left) / kTaskUnits);
        return split_time(full, left, (0.7 + 0.6 * fill) * slabs + 10, (0.35 + 0.75 * fill) * slabs + 3);
    };
    const double values = (double)s.tokens * s.H + (s.swiglu ? 3.0 : 2.0) * s.experts * s.I * s.H;
    return values * 10 / 6.2e6 + 15 + launch(s.columns_up(), s.H) + launch(s.columns_down(), s.I);
}
// ... on the 128 x 128 fp32 tile: 0.066 us a step of k and tile; as two launches, or where there are enough tasks on the queue, which
// fills whole rounds but for half a one and costs the more the more tokens there are.
inline double f32_tile_us(const PieceShape& s) {
    const SplitBlocks n = s.capped() ? exact_blocks(s.capacity, s.experts) : piece_blocks(s.pairs, s.experts);
    const int up = s.swiglu ? (s.I + 63) / 64 : (s.I + 127) / 128, down = (s.H + 127) / 128;
    const double t0 = n.small * up, t1 = n.small * down;
    const int64_t tasks = std::max<int64_t>(s.pairs / 128 + 1, std::min<int64_t>(s.pairs, s.experts)) * (up + down);
    if (s.experts > 1 && tasks >= 8 * kTaskUnits) return 0.066 * ((t0 * s.H + t1 * s.I) / kTaskUnits + 0.5 * std::max(s.H, s.I)) + 90;
    return 0.066 * (std::ceil(t0 / kTaskUnits) * s.H + std::ceil(t1 / kTaskUnits) * s.I) + 25;
}
// Whole layers, us, pieces / fp32 tile.  Enough rows to repay the pieces of the weights: the reference's knob file (8192 rows, one expert of
// 1024 x 4096, ReLU) 711 / 1067, 2048 rows of it 383 / 426; 8 experts of 1024 x 2048, GELU, 512 rows each 436 / 535; 16 of 2048 x 1408, SwiGLU, 512
// rows 1188 / 1298, 2048 rows 3186 / 4688; 8 of 512 x 1024, 768 rows 172 / 187; 2 of 4096 x 4096, 512 rows 791 / 1091.  A round of tasks that
// does not fill the chip either way: one of 1024 x 1024, 4096 rows 202 / 187, 8192 rows 238 / 315; one of 4096 x 4096, 1024 rows 697 / 572, 1536
// rows 712 / 1055.  Of 177 layers without binding drops (512 to 8192 rows an expert, half of them random shapes) the estimate takes the faster
// way at all but those nearer than 2 %.
// Where dropping binds, every token is still routed and taken apart, row blocks are chosen and launched for rows that are not there, and
// an expert's rows fill the fp32 tile's blocks: the estimate has to promise a tenth and 40 us.  8 of 1024 x 2048, GELU, at most 512 rows of 640
// 433 / 318, of 1024 505 / 322; at most 640 of 800 441 / 510, of 1280 509 / 521; 4 of 1024 x 4096, ReLU, 512 of 1024 550 / 439, 1536 of 1920
// 739 / 1051; 16 of 2048 x 2048, ReLU, 256 of 512 901 / 633, 512 of 640 964 / 1238; 8 of 512 x 1024, GELU, 1024 of 2048 267 / 187, 1536 of 1920
// 225 / 298.  Of 184 such layers (a quarter of them random) it takes the other way at 12, by 3 to 10 %; by the rows in front of
// the dropping alone 49 were slower than the tile, up to twice its time.
inline bool pieces_pay(const PieceShape& s) {
    const double pieces = pieces_us(s), tile = f32_tile_us(s);
    return s.capped() ? 1.1 * pieces + 40 < tile : pieces < tile;
}

}  // namespace moe355
