// The rule that takes fp32 layers to bf16 pieces, at layers that were measured both ways.
// Built with g++ under AddressSanitizer + UndefinedBehaviorSanitizer.
#include <cmath>
#include <cstdio>

#include "f32_pieces_choice.hpp"

using namespace moe355;

static int failed = 0;
static void check(bool want, int experts, int H, int I, bool swiglu, int64_t rows, int64_t capacity, int per_token = 1) {
    const PieceShape s{rows * experts / per_token, rows * experts, experts, H, I, swiglu, capacity ? capacity : rows * experts};
    if (pieces_pay(s) == want) return;
    ++failed;
    std::printf("FAILED: %d for %d experts of %d x %d, %lld rows, capacity %lld, swiglu %d (%.0f, %.0f us)\n", !want, experts, H, I, (long long)rows,
                (long long)capacity, swiglu, pieces_us(s), f32_tile_us(s));
}

int main() {
    // none dropped: faster at nearly all sizes ...
    check(true, 1, 1024, 4096, false, 8192, 0);
    check(true, 1, 1024, 4096, false, 2048, 0);
    check(true, 8, 1024, 2048, false, 512, 0);
    check(true, 16, 2048, 1408, true, 512, 0, 2);
    check(true, 16, 2048, 1408, true, 2048, 0, 2);
    check(true, 2, 4096, 4096, false, 512, 0);
    check(true, 8, 512, 1024, false, 768, 0, 2);
    // ... but for part of a round of tasks either way
    check(false, 1, 1024, 1024, false, 4096, 0);
    check(true, 1, 1024, 1024, false, 8192, 0);
    check(false, 1, 4096, 4096, false, 1024, 0);
    check(true, 1, 4096, 4096, false, 1536, 0);
    // a capacity that does not bind changes nothing
    check(true, 8, 1024, 2048, false, 512, 640);
    check(true, 8, 1024, 2048, false, 512, 512);
    // dropping binds: by the rows that are kept
    check(false, 8, 1024, 2048, false, 640, 512);
    check(false, 8, 1024, 2048, false, 1024, 512);
    check(true, 8, 1024, 2048, false, 800, 640);
    check(true, 8, 1024, 2048, false, 1536, 768);
    check(false, 4, 1024, 4096, false, 1024, 512);
    check(true, 4, 1024, 4096, false, 1920, 1536);
    check(false, 16, 2048, 2048, false, 512, 256, 2);
    check(true, 16, 2048, 2048, false, 640, 512, 2);
    check(false, 8, 512, 1024, false, 2048, 1024, 2);
    check(true, 8, 512, 1024, false, 1920, 1536, 2);
    check(false, 8, 2048, 2048, true, 512, 256, 2);
    check(true, 8, 2048, 2048, true, 1280, 1024, 2);
    // the ends of the range: finite, and no capacity is too small to ask about
    for (int experts : {1, 512})
        for (int64_t rows : {(int64_t)1, (int64_t)1 << 20})
            for (int64_t capacity : {(int64_t)1, rows * experts})
                for (int dim : {128, 65536}) {
                    const PieceShape s{rows * experts, rows * experts, experts, dim, 128, true, capacity};
                    if (std::isfinite(pieces_us(s)) && std::isfinite(f32_tile_us(s)) && pieces_us(s) > 0 && f32_tile_us(s) > 0) continue;
                    ++failed;
                    std::printf("FAILED: estimate for %d experts of %d, %lld rows, capacity %lld\n", experts, dim, (long long)rows, (long long)capacity);
                }
    std::printf("pieces: %d failed checks\n", failed);
    return failed ? 1 : 0;
}
