// The rules that choose between operands as stored and transposed copies, at products that were measured both ways.
// Built with g++ under AddressSanitizer + UndefinedBehaviorSanitizer.
#include <cstdio>

#include "product_choice.hpp"

using namespace moe355;

static int failed = 0;
static void check(bool got, bool want, const char* rule, int64_t A, int E, int N, int K) {
    if (got == want) return;
    ++failed;
    std::printf("FAILED %s: %d for %d experts of %d x %d, %lld rows\n", rule, got, E, N, K, (long long)A);
}
static void wgrad(bool want, int E, int N, int K, int rows) {
    const int64_t A = (int64_t)rows * E;
    check(wgrad_as_stored(A, E, N, K), want, "weight gradient", A, E, N, K);
    check(wgrad_as_stored(A, E, K, N), want, "weight gradient, other direction", A, E, K, N);
}

int main() {
    wgrad(true, 16, 2048, 2048, 512);
    wgrad(true, 16, 1408, 2048, 750);
    wgrad(true, 16, 1280, 1408, 136);
    wgrad(true, 16, 1024, 2560, 19);
    wgrad(true, 4, 2048, 2560, 4096);
    wgrad(true, 64, 1408, 2048, 1536);
    wgrad(false, 8, 4096, 2048, 2048);
    wgrad(false, 8, 4096, 14336, 512);
    wgrad(false, 8, 4096, 14336, 2048);
    // no hand-ordered tile behind the transposes: as stored, whatever that tile would take
    wgrad(true, 8, 960, 14336, 4096);
    wgrad(true, 64, 960, 4096, 2048);
    wgrad(true, 4, 960, 4096, 16384);
    wgrad(true, 12, 512, 512, 2000);
    // operands whose 32-bit offsets would wrap
    const int64_t rows = kBufferLimit / 2 / 4096;
    check(wgrad_as_stored(rows - 129, 8, 512, 4096), true, "largest operand", rows - 129, 8, 512, 4096);
    check(wgrad_as_stored(rows - 128, 8, 512, 4096), false, "operand of 4 GiB with its tile", rows - 128, 8, 512, 4096);
    check(grouped_kn_as_stored(rows - 128, 8, 512, 4096), false, "operand of 4 GiB with its tile", rows - 128, 8, 512, 4096);
    for (int E : {1, 512})
        for (int dim : {64, 65536})
            for (int64_t A : {(int64_t)1, (int64_t)1 << 30}) {
                const bool ok = stored_operands_ok(A, dim, 64);
                check(!wgrad_as_stored(A, E, dim, 64) || ok, true, "weight gradient at an end", A, E, dim, 64);
                check(!grouped_kn_as_stored(A, E, dim, 64) || ok, true, "data gradient at an end", A, E, dim, 64);
            }
    std::printf("product choice: %d failed checks\n", failed);
    return failed ? 1 : 0;
}
