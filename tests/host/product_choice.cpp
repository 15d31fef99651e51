// The rules that choose the tiles of a training step's products, at products that were measured both ways.
// Built with g++ under AddressSanitizer + UndefinedBehaviorSanitizer.
#include <cstdio>

#include "product_choice.hpp"

using namespace moe355;

static int failed = 0;
static void check(bool got, bool want, const char* rule, int64_t A, int E, int N, int K, int products = 1) {
    if (got == want) return;
    ++failed;
    std::printf("FAILED %s: %d for %d experts of %d x %d, %lld rows, %d products\n", rule, got, E, N, K, (long long)A, products);
}
static void wgrad(bool large, int products, int E, int N, int K, int rows) {
    const int64_t A = (int64_t)rows * E;
    check(wgrad_large(A, E, N, K, products), large, "weight gradient", A, E, N, K, products);
    check(wgrad_large(A, E, K, N, products), large, "weight gradient, other direction", A, E, K, N, products);
}
static void data(bool large, int products, int E, int N, int K, int rows) {
    const int64_t A = (int64_t)rows * E;
    check(grouped_kn_large(A, E, N, K, products), large, "data gradient", A, E, N, K, products);
}

int main() {
    // the large tile: whole rounds of it, long sums
    wgrad(true, 1, 16, 2048, 2048, 512);
    wgrad(true, 2, 16, 2048, 2048, 512);
    wgrad(true, 3, 16, 2048, 1408, 750);
    wgrad(true, 1, 4, 2048, 2560, 4096);
    wgrad(true, 1, 16, 2048, 2560, 1024);
    wgrad(true, 1, 8, 4096, 2048, 2048);
    wgrad(true, 1, 8, 4096, 14336, 2048);
    wgrad(true, 3, 8, 4096, 4096, 300);
    wgrad(true, 1, 8, 960, 14336, 4096);
    wgrad(true, 3, 4, 1024, 1024, 3652);
    wgrad(true, 3, 64, 2304, 1408, 194);
    wgrad(true, 2, 32, 2688, 768, 861);
    // the small one: fewer tiles than compute units, short sums
    wgrad(false, 1, 1, 1024, 4096, 8192);
    wgrad(false, 1, 1, 1024, 1024, 16384);
    wgrad(false, 3, 1, 1024, 1024, 16384);
    wgrad(false, 1, 16, 2688, 2688, 31);
    wgrad(false, 1, 8, 1408, 1408, 280);
    wgrad(false, 3, 8, 896, 1152, 564);
    wgrad(false, 3, 3, 2944, 1152, 66);
    wgrad(false, 1, 12, 512, 512, 2000);
    // ... and tiles of an expert that the large one leaves on few XCDs
    wgrad(false, 2, 64, 384, 256, 112);
    wgrad(false, 2, 64, 512, 256, 148);
    wgrad(false, 1, 12, 1408, 640, 132);
    wgrad(false, 3, 12, 512, 512, 2000);
    // one product does not fill a round of it, three do
    wgrad(false, 1, 2, 1536, 1536, 8192);
    wgrad(true, 3, 2, 1536, 1536, 8192);
    wgrad(false, 1, 1, 2048, 2048, 16384);
    wgrad(true, 3, 1, 2048, 2048, 16384);
    // data gradients
    data(true, 1, 16, 2048, 2048, 512);
    data(true, 1, 16, 1408, 2048, 750);
    data(true, 1, 4, 2560, 2048, 4096);
    data(true, 2, 4, 2560, 2048, 4096);
    data(false, 1, 8, 1664, 1280, 250);
    data(false, 1, 16, 1920, 1152, 175);
    data(false, 1, 8, 2560, 1024, 750);
    data(false, 1, 4, 2560, 1024, 750);
    // operands whose 32-bit offsets would wrap
    const int64_t rows = kBufferLimit / 2 / 4096;
    check(stored_operands_ok(rows - 129, 512, 4096), true, "largest operand", rows - 129, 8, 512, 4096);
    check(stored_operands_ok(rows - 128, 512, 4096), false, "operand of 4 GiB with its tile", rows - 128, 8, 512, 4096);
    // the ends of the range: an answer, and no overflow on the way to it
    for (int E : {1, 512})
        for (int dim : {64, 65536})
            for (int64_t A : {(int64_t)1, (int64_t)1 << 30})
                for (int products = 1; products <= 3; ++products) {
                    (void)wgrad_large(A, E, dim, 64, products);
                    (void)wgrad_large(A, E, dim, 65536, products);
                    if (A < ((int64_t)1 << 24)) (void)grouped_kn_large(A, E, dim, 64, products);
                }
    std::printf("product choice: %d failed checks\n", failed);
    return failed ? 1 : 0;
}
