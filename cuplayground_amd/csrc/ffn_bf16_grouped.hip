// Products on the 16-bit tiles (ffn_bf16_tile.hpp) outside the layer: dense operands, packed rows by expert, weight gradients.
#include <algorithm>

#include "ffn_bf16_tile.hpp"

namespace moe355 {
namespace {

// The bare reference contract on dense operands: rows [b*BM, ...) of A, one "expert".
template <class T>
__global__ __launch_bounds__(T::THREADS) void gemm_dense_kernel(const uint16_t* A, const uint16_t* B,
                                                                const uint16_t* bias, uint16_t* C, int M, int N, int K,
                                                                int act) {
    extern __shared__ __align__(16) unsigned char smem[];
    TaskPtrs p;
    const int row0 = blockIdx.x * T::BM;      // row tiles fastest: neighbouring workgroups share the weight tile
    p.a_base = A;
    p.gather = nullptr;
    p.a_row0 = row0;
    p.a_ld = K;
    p.b0 = B;
    p.b1 = nullptr;
    p.bias0 = bias;
    p.bias1 = nullptr;
    p.c_base = C + (int64_t)row0 * N;
    p.N = N;
    p.K = K;
    p.b_ld = K;
    p.rows = min(T::BM, M - row0);
    p.n0 = blockIdx.y * T::BN;
    p.act = act;
    p.swiglu = false;
    p.publish = false;
    p.a_extent = (uint32_t)((int64_t)M * K * 2);
    p.b_extent = (uint32_t)((int64_t)N * K * 2);
    p.part = nullptr; p.part_cnt = nullptr; p.kparts = 1; p.kpart = 0; p.poison = false;
    p.deriv = 0; p.aux0 = nullptr; p.aux1 = nullptr; p.c1_base = nullptr;
    gemm_tile<T>(p, smem);
}

// The tiles a grouped product runs on.  256: blocks of 256 rows, and of 128 where an expert has no more than that many rows left
// (the smaller tile takes 0.65 of the larger one's time; the other half of the larger one would multiply zeros).
template <bool F16_, int BIG_>
struct RowSplit {
    static constexpr bool F16 = F16_, HAND = true;
    static constexpr int BIG = BIG_, BN = 256, THREADS = 256;
    using TB = typename std::conditional<BIG_ == 256, Tile<256, 256, 2, 2, 2, F16_>, Tile<128, 256, 1, 4, 2, F16_>>::type;
    using TH = Tile<128, 256, 1, 4, 2, F16_>;
    static constexpr int LDS_BYTES = TB::LDS_BYTES;
    static_assert(TH::LDS_BYTES <= LDS_BYTES, "one dynamic LDS block for both");
};
// The 128 x 128 tile of the general loop.
template <bool F16_>
struct PlainSplit {
    static constexpr bool F16 = F16_, HAND = false;
    using TB = Tile<128, 128, 2, 2, 2, F16_>;
    static constexpr int BIG = 128, BN = 128, THREADS = 256, LDS_BYTES = TB::LDS_BYTES;
};

struct GroupedTask {
    int expert, row0, rows, ctile;
};
// Which tile workgroup `id` of a grouped product takes, from the experts' row counts alone; false: none.  Order: the row blocks of
// full height, expert by expert, column tile by column tile, an expert's row blocks fastest (neighbouring workgroups share a
// weight tile, an expert's few row blocks stay in the caches while its column tiles pass by); with 256-row blocks, behind them the
// remainders of at most 128 rows: the long tasks start first, and the short ones fill the compute units that the last round of
// long ones leaves idle.  Every wavefront works it out for itself, an expert a lane, which takes less time than a launch
// in front that writes tables.
// 16 experts of 2048 x 2048, 512 rows each, bf16: 112 -> 93 us (320 tasks on 256 compute units, 64 of them remainders); 8 of
// 4096 x 2048, 2048 rows 297 -> 258; 64 of 2048 x 1408, 94 rows 113 -> 106; 16 of 2048 x 1408, 750 rows, no remainders, 109 -> 110.
template <int BIG>
__device__ __forceinline__ bool grouped_task(const int32_t* __restrict__ count, const int32_t* __restrict__ offset, int E, int ncol, int id, GroupedTask& t) {
    constexpr int LEFT = BIG == 256 ? 128 : 0;          // rows up to which what is left of an expert is a block of its own kind
    const int lane = threadIdx.x & 63;
    auto rows_of = [&](int c) { return c + lane < E ? max(count[c + lane], 0) : 0; };
    auto big_of = [&](int n) { return (n + BIG - 1 - LEFT) / BIG; };
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
            const int local = id - first * ncol;
            t.ctile = local / blocks;
            const int rb = local - t.ctile * blocks;
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
// What a grouped product does with its sums: one kernel each, so that a tile's code is a slab loop and one epilogue (with three of
// them a kernel of several tiles is twice the instruction cache).
enum : int { kSums = 0, kGelu = 2, kDeriv = 4 };      // sums or ReLU; GELU; the activation's derivative
template <class T, int EPI>
__device__ __forceinline__ void grouped_epilogue(const TaskPtrs& p, unsigned char* smem, f32x4 (&acc)[T::TM][T::TN]) {
    epilogue_full_n_impl<T, EPI == kDeriv ? 0 : EPI, NoHook, WholeTile, EPI == kDeriv>(p, smem, acc, NoHook());
}
template <class P, int EPI>
__device__ __forceinline__ void grouped_tile(const TaskPtrs& p, unsigned char* smem) {
    if constexpr (!P::HAND) {
        static_assert(EPI != kDeriv, "the derivative lives in the epilogue of the hand-ordered tiles");
        gemm_tile<typename P::TB>(p, smem);
    } else {
        auto ring = [&](auto tile) {
            using T = decltype(tile);
            const RingLoads L = ring_prepare<T>(p);
            ring_first_loads<T>(L, smem);
            f32x4 acc[T::TM][T::TN];
            if (ring_slabs<T>(p.rows, L, smem, acc)) grouped_epilogue<T, EPI>(p, smem, acc);
        };
        if (P::BIG == 256 && p.rows > 128) ring(typename P::TB());
        else ring(typename P::TH());
    }
}

// Grouped GEMM on packed expert-major rows, outside the layer: out[r,:] = act(a[r,:] . w[e(r)]^T + bias[e(r)]) -- the
// reference's tile GEMM (mma.cuh:46-179) once per expert.  With the weight handed over in its K-major view this is the data
// gradient of a projection (dX = dY . W).  DERIV: that of the down projection with the activation's derivative in its epilogue,
// which hands on dU (and dG) instead of dH.  One workgroup per tile (grouped_task).
struct GroupedArgs {
    const uint16_t* a_rows;
    const uint16_t* w;
    const uint16_t* bias;        // or null
    const uint16_t* u_rows;      // DERIV: the saved projections ...
    const uint16_t* g_rows;      // ... and, with SwiGLU, the gate's
    uint16_t* out;               // rows of the result (DERIV: dU)
    uint16_t* out1;              // DERIV, SwiGLU: dG
    const int32_t* count;
    const int32_t* offset;
    int E, N, K, act;            // act: the epilogue's activation (DERIV: the layer's hidden_act)
    uint32_t a_bytes;
};
template <class P, int EPI>
__global__ __launch_bounds__(P::THREADS) void grouped_gemm_kernel(GroupedArgs a) {
    constexpr bool DERIV = EPI == kDeriv;
    extern __shared__ __align__(16) unsigned char smem[];
    const int N = a.N, K = a.K;
    GroupedTask t;
    if (!grouped_task<P::BIG>(a.count, a.offset, a.E, (N + P::BN - 1) / P::BN, blockIdx.x, t)) return;
    const int64_t at = (int64_t)t.row0 * N;
    TaskPtrs p;
    p.a_base = a.a_rows;
    p.gather = nullptr;
    p.a_row0 = t.row0;
    p.a_ld = K;
    p.b0 = a.w + (int64_t)t.expert * N * K;
    p.b1 = nullptr;
    p.b_ld = K;
    p.bias0 = a.bias ? a.bias + (int64_t)t.expert * N : nullptr;
    p.bias1 = nullptr;
    p.c_base = a.out + at;
    p.N = N;
    p.K = K;
    p.rows = t.rows;
    p.n0 = t.ctile * P::BN;
    p.act = DERIV ? MOE_ACT_NONE : a.act;
    p.swiglu = false;
    p.publish = false;
    p.a_extent = a.a_bytes;
    p.b_extent = (uint32_t)((int64_t)N * K * 2);
    p.part = nullptr; p.part_cnt = nullptr; p.kparts = 1; p.kpart = 0; p.poison = false;
    p.deriv = DERIV ? 1 + a.act : 0;
    p.aux0 = DERIV ? a.u_rows + at : nullptr;
    p.aux1 = DERIV && a.g_rows ? a.g_rows + at : nullptr;
    p.c1_base = DERIV && a.out1 ? a.out1 + at : nullptr;
    grouped_tile<P, EPI>(p, smem);
}

// Weight gradient of one projection: dw[e] [N, K] = dy_e^T . a_e, the sum running over the rows of expert e.  Both
// operands arrive transposed and padded: dyT [N, ld] and aT [K, ld] hold expert e's rows in columns
// [poff[e], poff[e+1]) (zeros behind the last real row; every window is a multiple of 128 wide), so each expert is one
// (M,K) x (N,K)^T tile GEMM over its window.  grid = (row tiles of N, column tiles of K, experts).
template <class T>
__global__ __launch_bounds__(T::THREADS) void wgrad_kernel(const uint16_t* dyT, const uint16_t* aT, uint16_t* dw,
                                                           const int32_t* poff, int N, int K, int ld, uint32_t dy_bytes,
                                                           uint32_t a_bytes) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int e = blockIdx.z;
    const int row0 = blockIdx.x * T::BM, n0 = blockIdx.y * T::BN;
    const int p0 = poff[e], window = poff[e + 1] - p0;
    uint16_t* c = dw + (int64_t)e * N * K + (int64_t)row0 * K;
    const int rows = min(T::BM, N - row0);
    if (window == 0) {   // an expert that received no rows: its gradient is zero
        for (int i = threadIdx.x; i < rows * T::BN; i += T::THREADS) {
            const int r = i / T::BN, col = n0 + i % T::BN;
            if (col < K) c[(int64_t)r * K + col] = 0;
        }
        return;
    }
    TaskPtrs p;
    p.a_base = dyT + p0;
    p.gather = nullptr;
    p.a_row0 = row0;
    p.a_ld = ld;
    p.b0 = aT + p0;
    p.b1 = nullptr;
    p.b_ld = ld;
    p.bias0 = nullptr;
    p.bias1 = nullptr;
    p.c_base = c;
    p.N = K;
    p.K = window;
    p.rows = rows;
    p.n0 = n0;
    p.act = MOE_ACT_NONE;
    p.swiglu = false;
    p.publish = false;
    p.a_extent = dy_bytes - (uint32_t)p0 * 2;
    p.b_extent = a_bytes - (uint32_t)p0 * 2;
    p.part = nullptr; p.part_cnt = nullptr; p.kparts = 1; p.kpart = 0; p.poison = false;
    p.deriv = 0; p.aux0 = nullptr; p.aux1 = nullptr; p.c1_base = nullptr;
    gemm_tile<T>(p, smem);
}

}  // namespace

template <class T>
static hipError_t launch_dense(const void* A, const void* B, const void* bias, void* C, int64_t M, int64_t N, int64_t K,
                               int act, hipStream_t st) {
    hipError_t e = allow_lds(&gemm_dense_kernel<T>, T::LDS_BYTES);
    if (e != hipSuccess) return e;
    const dim3 grid((unsigned)((M + T::BM - 1) / T::BM), (unsigned)((N + T::BN - 1) / T::BN));
    gemm_dense_kernel<T><<<grid, T::THREADS, T::LDS_BYTES, st>>>((const uint16_t*)A, (const uint16_t*)B,
                                                                 (const uint16_t*)bias, (uint16_t*)C, (int)M, (int)N,
                                                                 (int)K, act);
    return hipGetLastError();
}

hipError_t launch_gemm_dense_bf16(const void* A, const void* B, const void* bias, void* C, int64_t M, int64_t N,
                                  int64_t K, int act, int opt_tile, hipStream_t st, bool f16) {
    const int64_t lim = (int64_t)1 << 32;
    const bool large = M >= 1024 && N >= 1024 && N % 256 == 0 && K % 128 == 0 && M * K * 2 < lim && N * K * 2 < lim;
    {   // the tile asked for: 1 = 256 x 256, 2 = 128 x 256 (shapes they accept only), 0 = 128 x 128
        const int v = opt_tile;
        if (v == 0) return f16 ? launch_dense<Tile128H>(A, B, bias, C, M, N, K, act, st) : launch_dense<Tile128>(A, B, bias, C, M, N, K, act, st);
        if ((v == 1 || v == 2) && N % 256 == 0 && K % 128 == 0 && M * K * 2 < lim && N * K * 2 < lim) {
            if (v == 1) return f16 ? launch_dense<Tile256H>(A, B, bias, C, M, N, K, act, st) : launch_dense<Tile256>(A, B, bias, C, M, N, K, act, st);
            return f16 ? launch_dense<Tile128x256H>(A, B, bias, C, M, N, K, act, st) : launch_dense<Tile128x256>(A, B, bias, C, M, N, K, act, st);
        }
    }
    if (f16)
        return large ? launch_dense<Tile256H>(A, B, bias, C, M, N, K, act, st)
                     : launch_dense<Tile128H>(A, B, bias, C, M, N, K, act, st);
    return large ? launch_dense<Tile256>(A, B, bias, C, M, N, K, act, st)
                 : launch_dense<Tile128>(A, B, bias, C, M, N, K, act, st);
}

// ---- building blocks of the backward pass (callers: csrc/backward.hip) ----
bool grouped_hand_ok(int64_t A, int N, int K) { return A * K * 2 < kBufferLimit && hand_weights_ok(N, K); }
// Tile of one grouped product, as for a layer: 1, 2, or 0 when an operand has 4 GiB or more.
int grouped_gemm_tile_16(int64_t A, int E, int N, int K) {
    if (!grouped_hand_ok(A, N, K)) return 0;
    const int e = E > 0 ? E : 1;
    return projection_cost(true, A, e, columns256(N), K) <= projection_cost(false, A, e, columns256(N), K) ? 1 : 2;
}

template <class P, int EPI>
static hipError_t launch_grouped(const GroupedArgs& g, int64_t A, hipStream_t st) {
    const auto kernel = &grouped_gemm_kernel<P, EPI>;
    hipError_t e = allow_lds(kernel, P::LDS_BYTES);
    if (e != hipSuccess) return e;
    const int64_t blocks = (A / P::BIG + g.E) * ((g.N + P::BN - 1) / P::BN);      // no expert has more than rows / BIG + 1 row blocks
    if (blocks > INT32_MAX) return hipErrorInvalidValue;
    kernel<<<(unsigned)blocks, P::THREADS, P::LDS_BYTES, st>>>(g);
    return hipGetLastError();
}
template <bool F16, int EPI>
static hipError_t launch_grouped_tile(const GroupedArgs& g, int tile, int64_t A, hipStream_t st) {
    if (tile == 1) return launch_grouped<RowSplit<F16, 256>, EPI>(g, A, st);
    if (tile == 2) return launch_grouped<RowSplit<F16, 128>, EPI>(g, A, st);
    if constexpr (EPI != kDeriv) return launch_grouped<PlainSplit<F16>, EPI>(g, A, st);
    return hipErrorInvalidValue;
}

// tile: 1 (256-row blocks), 2 (128-row blocks) or 0 (the 128 x 128 tile of the general loop).
hipError_t launch_grouped_gemm_16(const void* a_rows, const void* w, const void* bias, void* out, const int32_t* count,
                                  const int32_t* offset, int tile, int64_t A, int E, int N, int K, int act, bool f16, hipStream_t st) {
    const GroupedArgs g{(const uint16_t*)a_rows, (const uint16_t*)w, (const uint16_t*)bias, nullptr, nullptr, (uint16_t*)out, nullptr,
                        count, offset, E, N, K, act, (uint32_t)(A * K * 2)};
    if (act == MOE_ACT_GELU) return f16 ? launch_grouped_tile<true, kGelu>(g, tile, A, st) : launch_grouped_tile<false, kGelu>(g, tile, A, st);
    return f16 ? launch_grouped_tile<true, kSums>(g, tile, A, st) : launch_grouped_tile<false, kSums>(g, tile, A, st);
}

// tile: 1 or 2: the hand-ordered tiles and those for their remainders only.
hipError_t launch_grouped_gemm_deriv_16(const void* a_rows, const void* w, const void* u, const void* g_rows, void* du, void* dg,
                                        const int32_t* count, const int32_t* offset, int tile, int64_t A, int E, int N, int K,
                                        int hidden_act, bool f16, hipStream_t st) {
    const GroupedArgs g{(const uint16_t*)a_rows, (const uint16_t*)w, nullptr, (const uint16_t*)u, (const uint16_t*)g_rows, (uint16_t*)du,
                        (uint16_t*)dg, count, offset, E, N, K, hidden_act, (uint32_t)(A * K * 2)};
    return f16 ? launch_grouped_tile<true, kDeriv>(g, tile, A, st) : launch_grouped_tile<false, kDeriv>(g, tile, A, st);
}

template <class T>
static hipError_t launch_wgrad(const void* dyT, const void* aT, void* dw, const int32_t* poff, int E, int N, int K,
                               int64_t ld, hipStream_t st) {
    hipError_t e = allow_lds(&wgrad_kernel<T>, T::LDS_BYTES);
    if (e != hipSuccess) return e;
    const dim3 grid((unsigned)((N + T::BM - 1) / T::BM), (unsigned)((K + T::BN - 1) / T::BN), (unsigned)E);
    wgrad_kernel<T><<<grid, T::THREADS, T::LDS_BYTES, st>>>((const uint16_t*)dyT, (const uint16_t*)aT, (uint16_t*)dw, poff,
                                                            N, K, (int)ld, (uint32_t)((int64_t)N * ld * 2),
                                                            (uint32_t)((int64_t)K * ld * 2));
    return hipGetLastError();
}

hipError_t launch_wgrad_16(const void* dyT, const void* aT, void* dw, const int32_t* poff, int E, int N, int K,
                           int64_t ld, bool f16, hipStream_t st) {
    const bool large = N >= 1024 && K >= 1024 && hand_weights_ok(N, ld) && hand_weights_ok(K, ld);
    if (large) return f16 ? launch_wgrad<Tile256H>(dyT, aT, dw, poff, E, N, K, ld, st)
                          : launch_wgrad<Tile256>(dyT, aT, dw, poff, E, N, K, ld, st);
    return f16 ? launch_wgrad<Tile128H>(dyT, aT, dw, poff, E, N, K, ld, st)
               : launch_wgrad<Tile128>(dyT, aT, dw, poff, E, N, K, ld, st);
}

}  // namespace moe355
