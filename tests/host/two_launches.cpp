// The rules that choose between the task queue and two launches, and between row blocks, at layers that were measured both ways.
// Built with g++ under AddressSanitizer + UndefinedBehaviorSanitizer.
#include <cstdio>
#include <cstdlib>

#include "two_launches.hpp"

using namespace moe355;

static int failed = 0;
static void check(bool got, bool want, const char* rule, const TwoLaunchShape& s) {
    if (got == want) return;
    ++failed;
    std::printf("FAILED %s: %d for %d experts of %d x %d, %lld rows, swiglu %d\n", rule, got, s.experts, s.H, s.I, (long long)s.pairs, s.swiglu);
}
static TwoLaunchShape shape(int experts, int H, int I, int rows, bool swiglu) { return TwoLaunchShape{(int64_t)rows * experts, experts, H, I, swiglu}; }
#define AUTO(want, large, drops, capacity, ...) check(two_launches_auto(shape(__VA_ARGS__), large, drops, capacity), want, "auto", shape(__VA_ARGS__))
#define ON256(want, ...) check(two_launches_on_256(shape(__VA_ARGS__)), want, "on 256", shape(__VA_ARGS__))
#define TABLE(want, ...) check(two_launches_keep_table(shape(__VA_ARGS__)), want, "table", shape(__VA_ARGS__))

int main() {
    // 128-row blocks: capped layers of few rows keep the queue
    AUTO(true, false, false, 1 << 20, 64, 2048, 1408, 29, true);
    AUTO(false, false, true, 38, 64, 2048, 1408, 38, true);
    AUTO(false, false, true, 48, 64, 2048, 1408, 48, true);
    AUTO(true, false, true, 49, 64, 2048, 1408, 49, true);
    // 256-row blocks: few rows an expert
    AUTO(true, true, false, 1 << 20, 64, 2048, 1408, 188, true);
    AUTO(true, true, true, 188, 64, 2048, 1408, 188, true);
    AUTO(false, true, false, 1 << 20, 32, 3456, 3264, 197, true);
    // ... many rounds: 11 of them, no drops
    AUTO(true, true, false, 1 << 20, 64, 2048, 1408, 1434, true);
    AUTO(false, true, false, 1 << 20, 64, 2048, 1408, 1024, true);
    AUTO(false, true, true, 1434, 64, 2048, 1408, 1434, true);
    AUTO(true, true, false, 1 << 20, 64, 4096, 1536, 956, true);
    AUTO(true, true, false, 1 << 20, 128, 1024, 1024, 1434, false);
    // ... and rows of eight experts that stay in the caches
    AUTO(false, true, false, 1 << 20, 32, 2048, 2048, 2867, false);
    AUTO(false, true, false, 1 << 20, 8, 4096, 14336, 5734, true);
    AUTO(false, true, false, 1 << 20, 16, 3072, 3072, 3823, false);
    // 256-row blocks under a plan of 128-row ones
    ON256(true, 18, 1856, 2944, 157, true);
    ON256(true, 17, 2048, 2048, 156, false);
    ON256(true, 9, 2048, 2112, 388, true);
    ON256(false, 64, 2048, 1408, 94, true);
    ON256(false, 16, 2048, 2048, 128, false);
    ON256(true, 64, 960, 896, 212, false);
    // ... the promised tenth, with a task's time from the length of its contraction
    ON256(false, 10, 1536, 1344, 297, true);
    ON256(false, 13, 1408, 1472, 212, true);
    ON256(false, 23, 768, 704, 143, true);
    ON256(false, 11, 1216, 768, 452, true);
    // the order of the row block table
    TABLE(true, 16, 2048, 2048, 262, true);
    TABLE(true, 16, 2048, 2048, 325, true);
    TABLE(false, 16, 2048, 2048, 237, true);
    TABLE(false, 16, 2048, 2048, 325, false);
    TABLE(false, 20, 2048, 3072, 290, false);
    TABLE(false, 64, 2048, 1408, 262, true);
    TABLE(true, 16, 3904, 1856, 306, true);
    TABLE(true, 8, 4032, 3968, 375, true);
    // ... nearly a round of long tasks
    TABLE(true, 8, 3264, 3392, 291, true);
    TABLE(true, 16, 4032, 3392, 356, false);
    TABLE(false, 16, 1920, 3136, 352, false);
    TABLE(false, 16, 1344, 3584, 316, false);
    TABLE(false, 16, 3840, 2944, 354, false);
    // ... with one or two experts an XCD only
    TABLE(false, 22, 1216, 2752, 309, false);
    TABLE(false, 24, 1024, 2560, 303, false);
    TABLE(false, 17, 1792, 3776, 346, false);
    TABLE(false, 48, 960, 1088, 297, false);
    // the ends of the range: every rule ends
    int answers = 0;
    for (int experts : {1, 512})
        for (int dim : {64, 65536})
            for (int64_t pairs : {(int64_t)1, (int64_t)1 << 30})
                for (bool swiglu : {false, true}) {
                    const TwoLaunchShape s{pairs, experts, dim, 65600 - dim, swiglu};
                    answers += two_launches_auto(s, true, false, pairs) + two_launches_on_256(s) + two_launches_keep_table(s) >= 0;
                }
    check(answers == 16, true, "the ends of the range", TwoLaunchShape{});
    std::printf("two launches: %d failed checks\n", failed);
    return failed ? 1 : 0;
}
