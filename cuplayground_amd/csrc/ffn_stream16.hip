// Expert FFN of bf16 / fp16 layers with a handful of token rows per expert (decoding): a weight streamer.
//
// Every weight of an expert that is hit is needed once, for a few rows: the time is the time the weights take from memory
// (8 experts of 4096 x 14336, SwiGLU, 16 tokens: 2.8 GB).  The 256-column tiles cannot reach that: a tile streams 256 weight
// rows through one compute unit's LDS behind one barrier per slab, and a down projection onto 4096 columns has 16 such tiles
// an expert, half the chip.  Here a wavefront is on its own:
//   * it owns 16 * CG output columns -- as many weight rows, or gate and up rows with SwiGLU -- over the whole contraction
//     dimension, as the "A" operand of v_mfma_f32_16x16x32; the "B" operand is up to NT groups of 16 token rows, read through
//     the caches that the neighbouring wavefronts read them through.  No LDS, no barrier;
//   * weights go from memory into the fragment registers in which the matrix instruction wants them (whole lines of eight rows
//     an instruction, two of which trade halves: stream_lines.hpp; 8 KB in flight while the 8 KB before are multiplied);
//   * one accumulator per output element, added to in the order of k as in the tiles: the same bits as theirs, and no sums
//     to bring together.
// A workgroup is four wavefronts on neighbouring columns of one row block.
//
// What bounds it: memory, and beside it the token rows, of which every wavefront reads NT * 16 for its 16 * CG weight rows.
// Measured, whole layer, cold weights, two launches, us -- 128 x 256 tile / NT 1, CG 1 / NT 2, CG 1 / NT 2, CG 2:
//   8 experts of 4096 x 14336, SwiGLU (2.8 GB): 2 rows each 507 / 438 / 468 / 445, 4 612 / 527 / 552 / 562,
//     8 613 / 556 / 579 / 566, 12 614 / 590 / 613 / 583, 16 618 / 823 / 657 / 609, 24 621 / 1237 / 740 / 648
//   16 of 2048 x 2048, GELU: 0.5 rows 96 / 50 / 54 / 67, 8 109 / 86 / 92 / 86, 12 108 / 103 / 97 / 88, 16 111 / 126 / 103 / 91,
//     24 111 / 149 / 128 / 117
//   64 of 2048 x 1408, SwiGLU: 2 rows 267 / 221 / 236 / 241, 8 284 / 264 / 276 / 261, 16 290 / 358 / 310 / 284, 24 294 / 468 / 349 / 309
//   12 of 1344 x 2752, GELU: 2 rows 105 / 63 / 69 / 76, 8 107 / 74 / 82 / 92, 16 106 / 102 / 92 / 99, 24 107 / 117 / 104 / 107
// (4 rows of the first: 5.7 TB/s of weights behind about 30 us of routing, launches and combine.)  An expert with more rows
// than a block had its weights read again for every block in these, which is where the steps upwards come from.  NT 4 was behind
// the tile from 24 rows on the first and the third of these.  Since then the weights come in whole lines and, where they are more than
// the memory-side cache holds, are not kept (stream_lines.hpp), us, before / this: 8 of 4096 x 14336, 0.25 rows each 177 / 171, 4 525 / 484, 10 586 /
// 509, 16 618 / 541; 64 of 2048 x 1408, 1.5 rows 193 / 175, 9 251 / 213, 16 269 / 231; 16 of 2048 x 2048, 2 rows 68 / 66.  The task queue with its written-through rows and pops
// of this much shorter tasks costs more than the overlap of the projections gives: 645 us against 520 (4 rows of the first),
// 158 against 81 (4 of the second).
//
// The form goes by the average; a skewed router gives some experts many times that.  Their blocks are taken up to 64 rows at a
// time, the token rows shared through LDS (take_group, stream_group).  Two launches, us -- 128 x 128 tile / every block by itself /
// groups, for router biases of 1 / rank^s:
//   64 experts of 2048 x 1408, top-6, 64 tokens: s = 0 338 / 254 / 253, 1.1 222 / 207 / 192, 2 137 / 157 / 136, one set of six 92 / 146 / 73;
//     96 tokens: 343 / 268 / 265, 233 / 245 / 201, 142 / 185 / 159, 96 / 170 / 112;  170: 348 / 283 / 283, 259 / 258 / 243, 169 / 192 / 173, 119 / 176 / 137
//   8 of 4096 x 14336, top-2, 32 tokens: 744 / 551 / 538, 745 / 686 / 619, 682 / 679 / 583, one set of two 362 / 352 / 292;
//     64 tokens: 748 / 610 / 610, 749 / 776 / 708, 687 / 755 / 674, 367 / 418 / 354
//   16 of 2048 x 2048, top-2, 64 tokens: 122 / 87 / 87, 117 / 92 / 91, 103 / 83 / 78;  128: 125 / 93 / 93, 123 / 127 / 115, 106 / 87 / 85
// (Groups of 64 rows in a wavefront's own fragments, without LDS, lose to single blocks: 890 us against 418 for 64 tokens on one set of two of the
// second; with one slab of weights on its way instead of two the groups take 469 there.)
// What is left behind the tile are routers that send nearly every one of 96 tokens and more to the same few of many experts.
#include "act_deriv.hpp"
#include "ffn_common.hpp"
#include "stream_lines.hpp"

namespace moe355 {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int STHREADS = 256;
constexpr int kGroupRows = 64, kGroupStage = kGroupRows * 128;      // rows of a group, bytes of 64 values of k of theirs

// COLD: the weights are too many for the caches: they are fetched once and not kept.
template <class ET, int NT, int CG, bool COLD_>
struct Stream {
    using Elem = ET;
    static constexpr bool COLD = COLD_;
    static constexpr bool F16 = std::is_same<ET, f16_s>::value;
    static constexpr int T = NT;             // groups of 16 token rows
    static constexpr int BM = 16 * NT;
    static constexpr int C = CG;             // groups of 16 columns a wavefront owns
    static constexpr int BN = 64 * CG;       // columns of a task
    static constexpr int WAVES = NT * CG > 1 ? 3 : 4;      // wavefronts per SIMD whose registers its own blocks leave room for
};

template <class P>
__device__ __forceinline__ f32x4 mfma32(u32x4 a, u32x4 b, f32x4 c) {
    if constexpr (P::F16) return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
template <class P>
__device__ __forceinline__ uint32_t pack2s(float lo, float hi) {
    if constexpr (P::F16) {
        typedef float f32x2_t __attribute__((ext_vector_type(2)));
        typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
        const f32x2_t v = {lo, hi};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2_t));
    } else {
        return pack2_bf16(lo, hi);
    }
}
template <class P>
__device__ __forceinline__ float widen1s(uint16_t v) {
    if constexpr (P::F16) return (float)__builtin_bit_cast(_Float16, v);
    else return bf16_bits_to_f32(v);
}

struct StreamTask {
    const uint16_t* w[2];      // weight matrices of the expert: {w_up or w_down, w_gate or null}
    const uint16_t* bias[2];
    const uint16_t* a_base;    // x or h
    const int32_t* gather;     // token_indices + row0, or null
    int64_t a_row0;
    uint16_t* c_base;          // h or y at the first row of the block
    int K, N, rows, n0, act;
    bool publish;              // rows are read by other workgroups of the same launch
};

// Bias, activation and the rows' store.  acc[m * CG + c][i]: matrix m, 16 columns c, 16 token rows i.
template <class P, int MATS, int NT>
__device__ __forceinline__ void stream_store(const StreamTask& t, int c0, f32x4 (&acc)[MATS * P::C][NT]) {
    constexpr int CG = P::C;
    const int lane = threadIdx.x & 63;
    const int idx = lane & 15, kg = lane >> 4;
    // this lane holds token rows 16 i + idx, columns c0 + 16 c + 4 kg ..+3
    const float relu_floor = t.act == MOE_ACT_RELU ? 0.0f : -INFINITY;      // compare and select: a NaN stays a NaN
#pragma unroll
    for (int c = 0; c < CG; ++c) {
        const int col = c0 + 16 * c + 4 * kg;
        float b[MATS][4];
#pragma unroll
        for (int m = 0; m < MATS; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) b[m][r] = t.bias[m] ? widen1s<P>(t.bias[m][col + r]) : -0.0f;
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            const int row = 16 * i + idx;
            if (row >= t.rows) continue;
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float u = acc[c][i][r] + b[0][r];
                if constexpr (MATS == 2) {
                    const float g = acc[CG + c][i][r] + b[1][r];
                    v[r] = silu16(g) * u;
                } else {
                    v[r] = t.act == MOE_ACT_GELU ? gelu16(u) : (u < relu_floor ? relu_floor : u);
                }
            }
            uint16_t* p = t.c_base + (int64_t)row * t.N + col;
            const uint32_t lo = pack2s<P>(v[0], v[1]), hi = pack2s<P>(v[2], v[3]);
            if (t.publish) publish8(p, lo, hi);
            else *reinterpret_cast<uint2*>(p) = uint2{lo, hi};
        }
    }
}

// MATS: weight matrices (2: SwiGLU's up and gate).  K and N are multiples of 64 (moe_config_validate), so a wavefront's
// columns exist together or not at all.
template <class P, int MATS>
__device__ __forceinline__ void stream_tile(const StreamTask& t) {
    constexpr int NT = P::T, CG = P::C, G = MATS * CG;
    constexpr int U = 8 / G;      // 32-wide slabs in flight
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int idx = lane & 15, kg = lane >> 4;
    const int c0 = t.n0 + 16 * CG * wave;
    if (c0 >= t.N) return;

    const char* wp[G];
#pragma unroll
    for (int g = 0; g < G; ++g) wp[g] = reinterpret_cast<const char*>(t.w[g / CG] + (int64_t)(c0 + 16 * (g % CG)) * t.K) + line_first(lane, 2 * (int64_t)t.K);
    const int64_t second = line_second(lane, 2 * (int64_t)t.K);
    // rows behind the block's last one read row 0 again and are never stored
    const uint16_t* xp[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const int r = 16 * i + idx < t.rows ? 16 * i + idx : 0;
        xp[i] = t.a_base + (t.gather ? (int64_t)t.gather[r] : t.a_row0 + r) * t.K + 8 * kg;
    }

    f32x4 acc[G][NT];
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int i = 0; i < NT; ++i) acc[g][i] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int slabs = t.K >> 5, full = slabs / U, left = slabs - full * U;
    u32x4 w[G][U], wn[G][U], x[NT][U];
    // slabs behind the last one read it again (and are not multiplied)
    auto load_w = [&](u32x4 (&d)[G][U], int s0) {
#pragma unroll
        for (int u = 0; u < U; u += 2) {       // (a line is two slabs; K is a multiple of 64, U even)
            const int k = min(s0 + u, slabs - 2) << 6;
#pragma unroll
            for (int g = 0; g < G; ++g) {
                d[g][u] = load_piece<P::COLD>(wp[g] + k);
                d[g][u + 1] = load_piece<P::COLD>(wp[g] + k + second);
            }
        }
    };
    auto settle = [&](int u) {
#pragma unroll
        for (int g = 0; g < G; ++g) line_pieces(w[g][u], w[g][u + 1], w[g][u], w[g][u + 1]);
    };
    auto load_x = [&](int s0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = min(s0 + u, slabs - 1) << 5;
#pragma unroll
            for (int i = 0; i < NT; ++i) x[i][u] = *reinterpret_cast<const u32x4*>(xp[i] + k);
        }
    };
    auto multiply = [&](int u) {
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int i = 0; i < NT; ++i) acc[g][i] = mfma32<P>(w[g][u], x[i][u], acc[g][i]);
    };
    load_w(w, 0);
    for (int c = 0; c < full; ++c) {
        // The token rows first: loads return in order, so waiting for them does not wait for the weights behind.
        load_x(c * U);
        if ((c + 1) * U < slabs) load_w(wn, (c + 1) * U);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; u += 2) {
            settle(u);
            multiply(u);
            multiply(u + 1);
        }
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int u = 0; u < U; ++u) w[g][u] = wn[g][u];
    }
    if (left) {
        load_x(full * U);
#pragma unroll
        for (int u = 0; u < U; u += 2)
            if (u < left) {
                settle(u);
                multiply(u);
                multiply(u + 1);
            }
    }

    stream_store<P, MATS, NT>(t, c0, acc);
}

template <class P>
__device__ __forceinline__ StreamTask resolve_stream(const FfnArgs& a, const Task& t, bool publish) {
    StreamTask p;
    const int64_t HI = (int64_t)a.H * a.I;
    p.publish = publish;
    p.rows = t.rows;
    p.n0 = t.ntile * P::BN;
    if (t.phase == 0) {
        const bool sw = a.act == MOE_ACT_SWIGLU;
        p.K = a.H;
        p.N = a.I;
        p.w[0] = (const uint16_t*)a.w_up + t.expert * HI;
        p.w[1] = sw ? (const uint16_t*)a.w_gate + t.expert * HI : nullptr;
        p.bias[0] = a.b_up ? (const uint16_t*)a.b_up + (int64_t)t.expert * a.I : nullptr;
        p.bias[1] = sw && a.b_gate ? (const uint16_t*)a.b_gate + (int64_t)t.expert * a.I : nullptr;
        p.a_base = (const uint16_t*)a.x;
        p.gather = a.token_indices + t.row0;
        p.a_row0 = 0;
        p.c_base = (uint16_t*)a.h + (int64_t)t.row0 * a.I;
        p.act = a.act;
    } else {
        p.K = a.I;
        p.N = a.H;
        p.w[0] = (const uint16_t*)a.w_down + t.expert * HI;
        p.w[1] = nullptr;
        p.bias[0] = a.b_down ? (const uint16_t*)a.b_down + (int64_t)t.expert * a.H : nullptr;
        p.bias[1] = nullptr;
        p.a_base = (const uint16_t*)a.h;
        p.gather = nullptr;
        p.a_row0 = t.row0;
        p.c_base = (uint16_t*)a.y + (int64_t)t.row0 * a.H;
        p.act = MOE_ACT_NONE;
    }
    return p;
}

// The same for up to 16 NT rows, more than a block has (take_group): the token rows go through LDS, 64 values of k at a time,
// once for the four wavefronts.  Weights as above, in the same order of k, hence the same bits.  Few workgroups have such a
// task, so nothing but a wavefront's own requests hides the memory's latency: two slabs of weights are always on their way,
// each requested as soon as the registers of the slab before the last are free.
template <class P, int MATS, int NT>
__device__ __forceinline__ void stream_group(const StreamTask& t, unsigned char* smem) {
    constexpr int CG = P::C, G = MATS * CG, PASSES = NT / 2;      // a pass brings 32 rows of 128 bytes
    constexpr int XD = G > 2 ? 1 : 2;            // slabs of rows in registers on their way to LDS (one: four weight fragments leave no room)
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int idx = lane & 15, kg = lane >> 4;
    const int c0 = t.n0 + 16 * CG * wave;
    const bool live = c0 < t.N;                  // a wavefront without columns helps to bring the rows
    // 32-bit offsets from bases that are the same in every lane: operands are below 4 GiB (large_tile_ok)
    const uint32_t w_off = (uint32_t)line_first(lane, 2 * (int64_t)t.K), w_second = w_off + (uint32_t)line_second(lane, 2 * (int64_t)t.K);
    uint32_t x_off[PASSES];
#pragma unroll
    for (int n = 0; n < PASSES; ++n) {
        const int row = (tid >> 3) + 32 * n, r = row < t.rows ? row : 0;      // rows behind the last one are never stored
        x_off[n] = (uint32_t)(((t.gather ? (int64_t)t.gather[r] : t.a_row0 + r) * t.K + 8 * (tid & 7)) * 2);
    }
    // 16-byte piece p of row r lies at p ^ (r >> 1 & 7): the 16 rows of a fragment read then meet all banks
    unsigned char* put = smem + (tid >> 3) * 128 + (((tid & 7) ^ ((tid >> 4) & 7)) << 4);
    const unsigned char* get = smem + idx * 128;
    const int sw = (idx >> 1) & 7;

    f32x4 acc[G][NT];
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int i = 0; i < NT; ++i) acc[g][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int slabs = t.K >> 6;
    u32x4 w[2][G][2], x[XD][PASSES];
    // slabs behind the last one read it again (and are not multiplied)
    auto load_x = [&](u32x4 (&d)[PASSES], int slab) {
        const char* base = reinterpret_cast<const char*>(t.a_base + (min(slab, slabs - 1) << 6));
#pragma unroll
        for (int n = 0; n < PASSES; ++n) d[n] = *reinterpret_cast<const u32x4*>(base + x_off[n]);
    };
    auto load_w = [&](u32x4 (&d)[G][2], int slab) {
        const int k = min(slab, slabs - 1) << 6;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const char* base = reinterpret_cast<const char*>(t.w[g / CG] + (int64_t)((live ? c0 : 0) + 16 * (g % CG)) * t.K + k);
            d[g][0] = load_piece<P::COLD>(base + w_off);
            d[g][1] = load_piece<P::COLD>(base + w_second);
        }
    };
    auto put_x = [&](const u32x4 (&d)[PASSES], int stage) {
#pragma unroll
        for (int n = 0; n < PASSES; ++n) *reinterpret_cast<u32x4*>(put + stage * kGroupStage + n * 32 * 128) = d[n];
    };
    // slab's rows lie in stage S; its successor's go into the other one, which was last read in front of the last barrier
    auto step = [&](auto S, int slab) {
        constexpr int st = decltype(S)::value;
#pragma unroll
        for (int g = 0; g < G; ++g) line_pieces(w[st][g][0], w[st][g][1], w[st][g][0], w[st][g][1]);
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int i = 0; i < NT; ++i) {
                const u32x4 b = *reinterpret_cast<const u32x4*>(get + st * kGroupStage + i * 16 * 128 + (((4 * u + kg) ^ sw) << 4));
#pragma unroll
                for (int g = 0; g < G; ++g) acc[g][i] = mfma32<P>(w[st][g][u], b, acc[g][i]);
            }
        __builtin_amdgcn_sched_barrier(0);
        put_x(x[(st ^ 1) % XD], st ^ 1);
        load_x(x[(st ^ 1) % XD], slab + 1 + XD);
        load_w(w[st], slab + 2);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
    };
    load_x(x[0], 0);
    load_w(w[0], 0);
    if constexpr (XD == 2) load_x(x[1], 1);
    load_w(w[1], 1);
    put_x(x[0], 0);
    load_x(x[0], XD);
    __syncthreads();
    for (int slab = 0; slab < slabs; slab += 2) {
        step(std::integral_constant<int, 0>{}, slab);
        if (slab + 1 < slabs) step(std::integral_constant<int, 1>{}, slab + 1);
    }
    if (live) stream_store<P, MATS, NT>(t, c0, acc);
}

// smem: null where a task never has more rows than a block.
template <class P, int MATS>
__device__ __forceinline__ void stream_rows(const StreamTask& p, unsigned char* smem) {
    if (!smem || p.rows <= P::BM) stream_tile<P, MATS>(p);
    else if (P::BM < 32 && p.rows <= 32) stream_group<P, MATS, 2>(p, smem);
    else stream_group<P, MATS, kGroupRows / 16>(p, smem);
}

template <class P>
__device__ __forceinline__ void stream_task(const FfnArgs& a, const Task& t, bool publish, unsigned char* smem) {
    const StreamTask p = resolve_stream<P>(a, t, publish);
    if (t.phase == 0 && a.act == MOE_ACT_SWIGLU) stream_rows<P, 2>(p, smem);
    else stream_rows<P, 1>(p, smem);
}

// The row blocks of an expert that was given more rows than a block holds, kGroupRows rows at a time: one block's task takes
// the group, the others have nothing to do (false).  The average that chooses the streamer says nothing about the fullest
// expert, and without this its weights are read again for every block.  Which block's varies with the column, because the
// blocks of a column are neighbours in the launch and go to the XCDs in turn: with the first one's, four blocks to an expert
// would leave the work to two of the eight XCDs.
template <class P>
__device__ __forceinline__ bool take_group(const FfnArgs& a, Task& t) {
    const Segment& s = a.seg_phase0[t.expert];
    constexpr int N = kGroupRows / P::BM;
    const int pos = t.mtile - s.mt0, first = pos / N * N, blocks = min(N, s.nmt - first);
    if (blocks == 1) return true;
    if (pos - first != (t.ntile * s.nmt >> 3) % blocks) return false;
    t.row0 -= (pos - first) * P::BM;
    t.rows = (blocks - 1) * P::BM + a.mtiles[s.mt0 + first + blocks - 1].rows;
    return true;
}

template <class P>
__global__ __launch_bounds__(STHREADS, P::WAVES) void ffn_tiled_stream16_kernel(FfnArgs a, int phase) {
    __shared__ int s_list[1 + kGroupRows];
    __shared__ __align__(16) unsigned char smem[2 * kGroupStage];
    if (phase == 0) zero_unrouted_rows(a, 2);
    Task t;
    if (!tiled_task(a, phase, blockIdx.x, t) || !take_group<P>(a, t)) return;
    stream_task<P>(a, t, phase == 1 && a.arrive, smem);
    if (phase == 1 && a.arrive) combine_arrivals<typename P::Elem>(combine_args(a), t.row0, t.rows, t.ntile, t.ntile * P::BN, P::BN, s_list);
}

template <class P>
__global__ __launch_bounds__(STHREADS) void ffn_persistent_stream16_kernel(FfnArgs a) {
    __shared__ int s_task, s_ok;
    __shared__ int s_cmb[kCombineLds];
    __shared__ int s_list[1 + P::BM];
    queue_kernel_entry();
    queue_clock_stamp(a.wg_clock, 0);
    zero_unrouted_rows(a, 2);
    const int ids = a.q->ids_queue;
    const int nseg = a.q->nseg;
    const int nnt0 = a.seg_phase0[0].nnt;
    QueueCursor cur = queue_cursor(a.groups);
    Task t;
    while (next_task(a, cur, &s_task, ids, nseg, nnt0, t)) {
        int ok = 1;
        if (t.phase == 1) ok = wait_phase0_done(a.done0, t.mtile, nnt0, a.spin_limit, a.q, a.host_stall, &s_ok);
        const long long started = trace_clock(a.task_trace);
        const bool publish = t.phase == 0 || publish_y(a);
        if (ok) {
            stream_task<P>(a, t, publish, nullptr);
        } else {
            const StreamTask p = resolve_stream<P>(a, t, publish);
            poison_tile(p.c_base, p.rows, p.N, p.n0, P::BN, 2);
        }
        if (a.task_trace) trace_task(a.task_trace, a.task_trace_cap, t.phase, t.expert, t.mtile, t.ntile, t.rows, started);
        if (t.phase == 0) signal_phase0_done(a.done0, t.mtile);
        else after_down_tile<typename P::Elem>(a, t.row0, t.rows, t.mtile, t.ntile, t.ntile * P::BN, P::BN, s_list);
    }
    if (a.combined) combine_while_idle_narrow<typename P::Elem>(sweep_args(a), &s_task, s_cmb);
    queue_clock_stamp(a.wg_clock, 1);
}

template <class P>
hipError_t launch(const FfnArgs& a, int max_mtiles, int nnt0, int nnt1, int blocks, hipStream_t st) {
    if (blocks > 0) {
        ffn_persistent_stream16_kernel<P><<<blocks, STHREADS, 0, st>>>(a);
    } else {
        ffn_tiled_stream16_kernel<P><<<tiled_grid(max_mtiles, nnt0, a.groups), STHREADS, 0, st>>>(a, 0);
        ffn_tiled_stream16_kernel<P><<<tiled_grid(max_mtiles, nnt1, a.groups), STHREADS, 0, st>>>(a, 1);
    }
    return hipGetLastError();
}

template <class P>
int occupancy() {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void*>(&ffn_persistent_stream16_kernel<P>), STHREADS, 0) != hipSuccess || n < 1)
        n = 1;
    return n;
}

}  // namespace

// The two forms: 0 = blocks of 16 rows, tasks of 64 columns; 1 = 32 rows, 128 columns.
template <class ET, bool COLD> using Narrow = Stream<ET, 1, 1, COLD>;
template <class ET, bool COLD> using Wide = Stream<ET, 2, 2, COLD>;

int stream16_block_m(int form) { return form ? Wide<bf16_s, true>::BM : Narrow<bf16_s, true>::BM; }
int stream16_block_n(int form) { return form ? Wide<bf16_s, true>::BN : Narrow<bf16_s, true>::BN; }
int ffn_persistent_occupancy_stream16(int form) { return form ? occupancy<Wide<bf16_s, true>>() : occupancy<Narrow<bf16_s, true>>(); }

template <class ET, bool COLD>
static hipError_t launch_form(const FfnArgs& a, int form, int max_mtiles, int nnt0, int nnt1, int blocks, hipStream_t st) {
    return form ? launch<Wide<ET, COLD>>(a, max_mtiles, nnt0, nnt1, blocks, st) : launch<Narrow<ET, COLD>>(a, max_mtiles, nnt0, nnt1, blocks, st);
}
// blocks > 0: workgroups of the task queue; 0: a launch per projection.
hipError_t launch_ffn_stream16(const FfnArgs& a, int form, bool f16, int max_mtiles, int nnt0, int nnt1, int blocks, hipStream_t st) {
    const bool cold = stream_cold(a, 2);
    if (f16) return cold ? launch_form<f16_s, true>(a, form, max_mtiles, nnt0, nnt1, blocks, st) : launch_form<f16_s, false>(a, form, max_mtiles, nnt0, nnt1, blocks, st);
    return cold ? launch_form<bf16_s, true>(a, form, max_mtiles, nnt0, nnt1, blocks, st) : launch_form<bf16_s, false>(a, form, max_mtiles, nnt0, nnt1, blocks, st);
}

}  // namespace moe355
