// Expert FFN for e4m3 weights with 128x128 block scales when every expert sees many token rows (prefill-sized
// batches of torch_dtype 4).  ffn_fp8.hip streams the weights once per 16-token row block, which is right for
// decode and wrong here: with hundreds of rows per expert each weight byte would be fetched again for every 16 rows.
// This file is the tile GEMM of the reference (mma.cuh:46-179: C = act(A.B^T + bias), A (M,K), B (N,K) row-major,
// fp32 accumulation, one cast on store) for that operand pair, with the numerics of ffn_fp8.hip:
//   y[n] = sum over 128-wide k blocks of scale[n/128][kb] * (fp32 dot product of that block).
//
// A task is (expert, 128-token row block, 128 weight rows): 64 gate + 64 up rows for a SwiGLU up projection (the pairs
// stay inside a lane), 128 rows of w_up for ReLU / GELU layers, 128 rows of w_down for the down projection; so all
// weight rows of a wavefront's fragments lie in one scale block and the scale of a k block is one scalar (two for a
// SwiGLU up projection).
//   * four wavefronts of 64 x 64 outputs, v_mfma_f32_16x16x32_bf16, weights as the "A" operand;
//   * K slabs of 64: token rows and weight bytes go from global memory straight into LDS (global_load ... lds), two slabs ahead, as
//     128- and 64-byte rows with xor-swizzled 16-byte chunks; weight bytes are widened to bf16 (exact) behind their fragment reads;
//   * a second accumulator set takes the 128-deep partial sums (its first MFMA of a k block starts from zero); after
//     every second slab acc = fma(scale, partial, acc) in fp32;
//   * three 24 KiB LDS stages per workgroup, two workgroups per compute unit.
#include <type_traits>

#include "ffn_common.hpp"

namespace moe355 {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void gbl_void;

constexpr int PBM = 128;          // token rows per row block
constexpr int PBN = 128;          // weight rows per tile
constexpr int PN0 = 64;           // intermediate columns per up-projection task (64 gate + 64 up rows)
constexpr int PN1 = 128;          // output columns per down-projection task
constexpr int PBK = 64;           // k per slab
constexpr int PROW = 128;         // bytes per LDS row (64 bf16)
constexpr int PSTAGE = (PBM + PBN) * PROW;
constexpr int PLDS_M8 = 2 * PSTAGE + 2 * PBM * 4; // e4m3 x e4m3 loop: behind the two stages, the token rows' scales of either slab
constexpr int PWROW = 64;         // bytes per LDS row of the weights (64 e4m3)
constexpr int PLDS = 3 * (PBM * PROW + PBN * PWROW);
static_assert(PLDS >= 4 * (PBM / 2 * PROW + PBN * PWROW), "the ring of row blocks of at most 64 rows");
constexpr int PTHREADS = 256;
constexpr int PTM = 4, PTN = 4;   // 16 x 16 fragments per wavefront: tokens, weight rows
constexpr int PRW = PBN * 4 / PTHREADS;        // 16-byte weight loads (16 e4m3 values) per thread per slab

struct TileTask {
    const uint16_t* a_base;     // x or h
    const int32_t* gather;      // token_indices + row0, or null
    int64_t a_row0;
    const uint8_t* w[2];        // up projection: {w_gate, w_up} of the expert; down projection: {w_down, w_down}
    const float* s[2];          // their scale rows: &scale[expert][c0 / 128][0]
    const uint16_t* bias[2];
    uint16_t* c_base;           // h or y at the first row of the block
    int K, N, rows, c0, phase;
    int act;                    // up projection without SwiGLU: the activation of the epilogue (else MOE_ACT_NONE)
    bool paired;                // up projection with SwiGLU: 64 gate + 64 up rows; otherwise 128 rows of one matrix
    bool publish;               // rows are read by other workgroups of the same launch
    // e4m3 x e4m3 plan: the token operand as e4m3 codes (rows as a_base's: gathered or a_row0 + r) and its scales
    const uint8_t* aq;          // [*, K]
    const float* sa;            // [*, K / 128]
};

// 8 e4m3 bytes -> 8 bf16 (exact), two an instruction.
__device__ __forceinline__ bf16x8 widen8(uint32_t lo, uint32_t hi) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const bf16x2 a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, false), b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, true);
    const bf16x2 c = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, false), d = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, true);
    const u32x4 v = {__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, c), __builtin_bit_cast(uint32_t, d)};
    return __builtin_bit_cast(bf16x8, v);
}

// The slab loop.  What bounds it: the latency of its loads; a slab's MFMAs are 0.2 us on a SIMD, a load from beyond the L2 takes 1 us and
// more.  So both operands go from memory to LDS as they are stored, two slabs ahead, in a ring of three stages (two workgroups
// per compute unit), and the weight bytes are widened behind their fragment reads: twice per workgroup then (two wavefronts
// share weight rows), at two values an instruction, but without registers, LDS writes and waits for bytes on their way.
// Weight bytes through registers, widened once per workgroup and written to LDS, the token rows one slab ahead / this (with blocks of 64,
// below), whole layers, us: 8 experts of 4096 x 14336, SwiGLU, 50 rows each 530 / 425, 250 1055 / 962, 500 1867 / 1677, 1024 3517 / 3103; 64 of
// 7168 x 2048, 37 rows 860 / 701, 500 3757 / 3410; 16 of 2048 x 2048, 500 rows 362 / 329; 256 of 7168 x 2048, 46 rows 3420 / 2866.
// PARTIAL: the row block holds fewer than ROWS rows; fragments that lie entirely in the padding are skipped.  ROWS = 64: a stage is two
// thirds as large, so that the ring has four and the loads run three slabs ahead (such a block is bound by the weight bytes in
// flight), and its rows are shared by all four wavefronts.  Blocks of 128 for all /
// this, us: 8 experts of 4096 x 14336, 32 rows each 458 / 406, 50 478 / 425, 175 (128 + 47) 772 / 737; 64 of 7168 x 2048, 37 rows 775 / 701; 256 of
// them, 46 rows 3110 / 2866; without such blocks as before.
template <bool PARTIAL, int ROWS>
__device__ __forceinline__ void tile_mainloop(const TileTask& p, unsigned char* smem, f32x4 (&acc)[ROWS / 32][PTN]) {
    constexpr int TM = ROWS / 32;                  // 16 x 16 fragments of token rows per wavefront
    constexpr int AHEAD = ROWS == 64 ? 3 : 2;
    constexpr int LOADS_A = ROWS * 8 / PTHREADS;   // 16-byte token loads per thread per slab
    constexpr int STAGE = ROWS * PROW + PBN * PWROW;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;

    // token rows: 8 threads per 128-byte row.  LDS slot (row, c) holds what a lane of a fragment takes as "chunk c ^ ((row >> 1) & 7)":
    // a lane's 16 weight bytes are 16 values of k in a row, eight for either half of the slab, so chunk 4 s + f of the tokens is
    // the one of k = 16 f + 8 s.
    const int prow = tid >> 3;
    const int slot = (tid & 7) ^ ((prow >> 1) & 7);
    const int chunk = 2 * (slot & 3) + (slot >> 2);
    const uint16_t* a_src[LOADS_A];
#pragma unroll
    for (int i = 0; i < LOADS_A; ++i) {
        int r = prow + i * 32;
        if (r >= p.rows) r = 0;                                   // padding rows re-read row 0; never stored
        const int64_t src_row = p.gather ? (int64_t)p.gather[r] : p.a_row0 + r;
        a_src[i] = p.a_base + src_row * p.K + chunk * 8;
    }
    // weight rows: 4 threads per 64-byte row; slot c of row j holds chunk c ^ weight_swizzle(j).  The LDS serves a 16-byte read to lanes 0-3,
    // 12-15 and 20-27 in one cycle, to 4-11, 16-19 and 28-31 in the next (and so on): of rows four apart, which meet the same banks,
    // two take chunk f and two f ^ 1, and all four must differ.
    auto weight_swizzle = [](int row) { return (4 - (row >> 2)) & 3; };
    // (a wavefront's 16 rows are rows of one matrix: a scalar address, and one 32-bit offset for both loads)
    const int wave_u = __builtin_amdgcn_readfirstlane(wave), brow = tid >> 2;
    const uint8_t* b_src[PRW];
#pragma unroll
    for (int i = 0; i < PRW; ++i)         // paired: wavefront column i owns tile rows [64 i, 64 i + 64): 32 gate rows, then 32 up rows
        b_src[i] = (p.paired && (wave_u >> 1) ? p.w[1] : p.w[0]) + (int64_t)(p.c0 + i * (p.paired ? 32 : 64)) * p.K;
    const uint32_t b_lane = (uint32_t)(p.paired ? brow & 31 : brow) * (uint32_t)p.K + ((tid & 3) ^ weight_swizzle(brow)) * 16;

    const int awave = __builtin_amdgcn_readfirstlane(prow & ~7) * PROW, bwave = __builtin_amdgcn_readfirstlane((tid >> 2) & ~15) * PWROW;
    auto issue = [&](int kt, int stage) {
        unsigned char* st = smem + stage;
#pragma unroll
        for (int i = 0; i < LOADS_A; ++i)
            __builtin_amdgcn_global_load_lds((gbl_void*)(a_src[i] + kt * PBK), (lds_void*)(st + awave + i * 32 * PROW), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < PRW; ++i)
            __builtin_amdgcn_global_load_lds((gbl_void*)(b_src[i] + kt * PBK + b_lane), (lds_void*)(st + ROWS * PROW + bwave + i * 64 * PWROW), 16, 0, 0);
    };

    const int frow = lane & 15, fk = lane >> 4;
    const int sw = (frow >> 1) & 7;
    const int ta = PARTIAL ? min(TM, max(0, (p.rows - wm * 16 * TM + 15) >> 4)) : TM;
    const int a_off = (wm * 16 * TM + frow) * PROW;
    const int b_off = ROWS * PROW + (wn * 16 * PTN + frow) * PWROW + ((fk ^ weight_swizzle(frow)) << 4);      // (of rows 16 apart the swizzle is the same)

    f32x4 part[TM][PTN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < PTN; ++j) {
            acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
            part[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }

    // The scales are read-only for the whole launch: scalar loads through the constant address space, issued a k block
    // ahead of their use.
    typedef const __attribute__((address_space(4))) float cfloat;
    cfloat* sc0 = (cfloat*)(uintptr_t)p.s[0];
    cfloat* sc1 = (cfloat*)(uintptr_t)p.s[1];

    // One slab: fragments from LDS, two halves of TM x PTN MFMAs into the partial sums (FIRST: the first of a k block starts from zero).
    auto slab = [&](int stage, auto first_c) {
        constexpr bool FIRST = decltype(first_c)::value;
        const unsigned char* st = smem + stage;
        u32x4 raw[PTN];
#pragma unroll
        for (int j = 0; j < PTN; ++j) raw[j] = *reinterpret_cast<const u32x4*>(st + b_off + j * 16 * PWROW);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int c = ((s * 4 + fk) ^ sw) << 4;
            bf16x8 af[TM], bf[PTN];
#pragma unroll
            for (int i = 0; i < TM; ++i)
                if (!PARTIAL || i < ta) af[i] = *reinterpret_cast<const bf16x8*>(st + a_off + i * 16 * PROW + c);
#pragma unroll
            for (int j = 0; j < PTN; ++j) bf[j] = widen8(raw[j][2 * s], raw[j][2 * s + 1]);
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                if (PARTIAL && i >= ta) continue;
#pragma unroll
                for (int j = 0; j < PTN; ++j)
                    part[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[j], af[i], FIRST && s == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : part[i][j], 0, 0, 0);
            }
        }
    };
    // The next slab has landed (loads return in issue order; later: how many slabs behind it may still be on their way), and this
    // wavefront's reads of LDS are done; then a barrier without the fences of __syncthreads(), which would wait for every load.
    auto end_slab = [&](auto later) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(decltype(later)::value * (LOADS_A + PRW)) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    typedef std::integral_constant<int, 0> None;
    typedef std::integral_constant<int, AHEAD - 1> Behind;
    auto fold = [&](float s0, float s1) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < PTN; ++j) {
                const float sc = j < PTN / 2 ? s0 : s1;
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[i][j][r] = __builtin_fmaf(sc, part[i][j][r], acc[i][j][r]);
            }
    };
    // Stages are taken in turn: here slab kt's, ahead that of slab kt + AHEAD, which slab kt - 1 has left.
    auto next = [](int stage) { return stage == AHEAD * STAGE ? 0 : stage + STAGE; };
    int here = 0, ahead = AHEAD * STAGE;
    const int KT = p.K >> 6;                // even
    __syncthreads();                        // the previous task may still be reading the stages
#pragma unroll
    for (int kt = 0; kt < AHEAD; ++kt)
        if (kt < 2 || kt < KT) issue(kt, kt * STAGE);
    if (KT >= AHEAD) end_slab(Behind{});
    else end_slab(None{});
    int kt = 0;
    auto k_block = [&](auto more0_c, auto more1_c) {     // slabs kt + AHEAD and kt + 1 + AHEAD exist
        const float s0 = sc0[kt >> 1], s1 = sc1[kt >> 1];
        auto one = [&](auto half_c, auto more_c) {
            constexpr int half = decltype(half_c)::value;
            constexpr bool more = decltype(more_c)::value;
            if constexpr (more) issue(kt + half + AHEAD, ahead);
            slab(here, std::integral_constant<bool, half == 0>{});
            if constexpr (half == 1) fold(s0, s1);
            end_slab(std::integral_constant<int, more ? AHEAD - 1 : 0>{});
            here = next(here);
            ahead = next(ahead);
        };
        one(std::integral_constant<int, 0>{}, more0_c);
        one(std::integral_constant<int, 1>{}, more1_c);
        kt += 2;
    };
    typedef std::true_type Yes;
    typedef std::false_type No;
    while (kt + 1 + AHEAD < KT) k_block(Yes{}, Yes{});
    if constexpr (AHEAD == 3) {
        if (kt + AHEAD < KT) k_block(Yes{}, No{});
    }
    k_block(No{}, No{});
}

// ---- the same tile with both operands e4m3: v_mfma_f32_16x16x128_f8f6f4 ----
//
// One matrix instruction takes a whole 128-wide k block (32 bytes of each operand per lane), twice the rate of the 16-bit
// instructions, and nothing is widened: token rows arrive as e4m3 codes with one fp32 scale per (row, k block)
// (quant_rows128 passes in front of the two projections), weights are fed as stored.  A slab is one k block: 128 bytes
// per row, both operands global -> LDS directly, the 16-bit tiles' row layout (128-byte rows, 16-byte chunks xor-swizzled
// by (row >> 1) & 7); a lane's fragment is chunks fk and 4 + fk of its row -- the two chunks the 16-bit tiles read, a
// pattern without LDS bank conflicts; with chunks 2 fk and 2 fk + 1 every second cycle of the reads was one (which k a
// lane's bytes stand for inside the instruction does not matter as long as both operands agree: the block's dot product
// is a sum over all of them).
// Every MFMA starts from zero; its 16 x 16 partial sums are scaled by (weight block scale) x (token row scale) and added
// in fp32: y[t, n] = sum over k blocks of s_w[n / 128][kb] * s_a[t][kb] * (dot product of the block's codes).
typedef int i32x8 __attribute__((ext_vector_type(8)));

template <bool PARTIAL>
__device__ __forceinline__ void tile_mainloop_mfma8(const TileTask& p, unsigned char* smem, f32x4 (&acc)[PTM][PTN]) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int KB = p.K >> 7;

    // both operands: 8 threads per 128-byte row, four passes of 32 rows; LDS slot (row, c) holds chunk c ^ ((row >> 1) & 7)
    const int prow = tid >> 3;
    const int chunk = (tid & 7) ^ ((prow >> 1) & 7);
    const uint8_t* a_src[4];
    const uint8_t* b_src[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        int r = prow + i * 32;
        if (r >= p.rows) r = 0;                                   // padding rows re-read row 0; never stored
        const int64_t src_row = p.gather ? (int64_t)p.gather[r] : p.a_row0 + r;
        a_src[i] = p.aq + src_row * p.K + chunk * 16;
        const int j = prow + i * 32;                              // row of the weight tile
        const uint8_t* base = p.w[0];
        int col;
        if (p.paired) {       // wavefront column w owns tile rows [64 w, 64 w + 64): 32 gate rows, then 32 up rows
            const int w = j >> 6, jj = j & 63;
            col = p.c0 + w * 32 + (jj & 31);
            base = (jj >> 5) ? p.w[1] : p.w[0];
        } else {
            col = p.c0 + j;
        }
        b_src[i] = base + (int64_t)col * p.K + chunk * 16;
    }
    const int wrow = __builtin_amdgcn_readfirstlane(prow & ~7);
    // The scales of the slab's token rows travel like the slab, global -> LDS, one float per row (wavefronts 0 and 1: a row
    // per lane).  As register loads they sat between the slab's requests in the memory counter, and the wait the compiler
    // puts in front of their use waited for the next slab's requests as well: no request was in flight during a slab's
    // MFMAs (MFMA pipes busy 24 % of the time).
    float* const ssc = reinterpret_cast<float*>(smem + 2 * PSTAGE);        // [stage][PBM]
    const float* sc_src = nullptr;
    if (wave < 2) {
        int r = tid;
        if (r >= p.rows) r = 0;
        const int64_t src_row = p.gather ? (int64_t)p.gather[r] : p.a_row0 + r;
        sc_src = p.sa + src_row * KB;
    }
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    auto issue = [&](int kb) {
        unsigned char* sa = smem + (kb & 1) * PSTAGE;
        unsigned char* sb = sa + PBM * PROW;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            __builtin_amdgcn_global_load_lds((gbl_void*)(a_src[i] + kb * 128), (lds_void*)(sa + (wrow + i * 32) * PROW), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            __builtin_amdgcn_global_load_lds((gbl_void*)(b_src[i] + kb * 128), (lds_void*)(sb + (wrow + i * 32) * PROW), 16, 0, 0);
        if (wave_u < 2)
            __builtin_amdgcn_global_load_lds((gbl_void*)(sc_src + kb), (lds_void*)(ssc + (kb & 1) * PBM + wave_u * 64), 4, 0, 0);
    };

    const int frow = lane & 15, fk = lane >> 4;
    const int sw = (frow >> 1) & 7;
    const int ta = PARTIAL ? min(PTM, max(0, (p.rows - wm * 16 * PTM + 15) >> 4)) : PTM;
    const int a_off = (wm * 16 * PTM + frow) * PROW;
    const int b_off = PBM * PROW + (wn * 16 * PTN + frow) * PROW;
    const int c0 = (fk ^ sw) << 4, c1 = ((4 + fk) ^ sw) << 4;

    const int sc_off = wm * 16 * PTM + frow;          // this lane's token rows (one per 16 x 16 fragment) in a stage's scales
    typedef const __attribute__((address_space(4))) float cfloat;
    cfloat* sc0 = (cfloat*)(uintptr_t)p.s[0];
    cfloat* sc1 = (cfloat*)(uintptr_t)p.s[1];

#pragma unroll
    for (int i = 0; i < PTM; ++i)
#pragma unroll
        for (int j = 0; j < PTN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    auto frag = [&](const unsigned char* base) {
        const u32x4 lo = *reinterpret_cast<const u32x4*>(base + c0), hi = *reinterpret_cast<const u32x4*>(base + c1);
        return i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
    };

    __syncthreads();                        // the previous task may still be reading the stages
    issue(0);
    for (int kb = 0; kb < KB; ++kb) {
        // slab kb has landed (it was requested a whole slab ago, and nothing younger is outstanding that we could let
        // fly: wait for all), and every wavefront is done reading the other stage
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (kb + 1 < KB) issue(kb + 1);
        float sac[PTM];
#pragma unroll
        for (int i = 0; i < PTM; ++i) sac[i] = ssc[(kb & 1) * PBM + sc_off + i * 16];
        const float s0 = sc0[kb], s1 = sc1[kb];
        const unsigned char* st = smem + (kb & 1) * PSTAGE;
        i32x8 bf[PTN];
#pragma unroll
        for (int j = 0; j < PTN; ++j) bf[j] = frag(st + b_off + j * 16 * PROW);
#pragma unroll
        for (int i = 0; i < PTM; ++i) {
            if (PARTIAL && i >= ta) continue;
            const i32x8 af = frag(st + a_off + i * 16 * PROW);
            const float m0 = s0 * sac[i], m1 = s1 * sac[i];
#pragma unroll
            for (int j = 0; j < PTN; ++j) {
                const f32x4 part = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bf[j], af, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
                const float m = j < PTN / 2 ? m0 : m1;
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[i][j][r] = __builtin_fmaf(m, part[r], acc[i][j][r]);
            }
        }
    }
}

// acc[i][j][r]: token row = 16 (TM wm + i) + (lane & 15); weight row inside fragment j = 4 (lane >> 4) + r.
template <int TM>
__device__ __forceinline__ void tile_epilogue(const TileTask& p, f32x4 (&acc)[TM][PTN]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int frow = lane & 15, fk = lane >> 4;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int m = wm * 16 * TM + i * 16 + frow;
        if (m >= p.rows) continue;
        uint16_t* crow = p.c_base + (int64_t)m * p.N;
        if (p.paired) {
#pragma unroll
            for (int j = 0; j < PTN / 2; ++j) {
                const int col = p.c0 + wn * 32 + j * 16 + 4 * fk;
                float o[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float g = acc[i][j][r], u = acc[i][j + PTN / 2][r];
                    if (p.bias[0]) g = g + bf16_bits_to_f32(p.bias[0][col + r]);
                    if (p.bias[1]) u = u + bf16_bits_to_f32(p.bias[1][col + r]);
                    o[r] = silu(g) * u;
                }
                const uint32_t lo = pack2_bf16(o[0], o[1]), hi = pack2_bf16(o[2], o[3]);
                if (p.publish) publish8(crow + col, lo, hi);
                else *reinterpret_cast<uint2*>(crow + col) = uint2{lo, hi};
            }
        } else {
#pragma unroll
            for (int j = 0; j < PTN; ++j) {
                const int col = p.c0 + wn * 64 + j * 16 + 4 * fk;
                float o[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    o[r] = acc[i][j][r];
                    if (p.bias[0]) o[r] = o[r] + bf16_bits_to_f32(p.bias[0][col + r]);
                    o[r] = act_apply(o[r], p.act);
                }
                const uint32_t lo = pack2_bf16(o[0], o[1]), hi = pack2_bf16(o[2], o[3]);
                if (p.publish) publish8(crow + col, lo, hi);
                else *reinterpret_cast<uint2*>(crow + col) = uint2{lo, hi};
            }
        }
    }
}

__device__ __forceinline__ void fp8_gemm_tile(const TileTask& p, unsigned char* smem) {
    if (p.rows <= PBM / 2) {
        f32x4 acc[PTM / 2][PTN];
        tile_mainloop<true, PBM / 2>(p, smem, acc);
        tile_epilogue(p, acc);
        return;
    }
    f32x4 acc[PTM][PTN];
    if (p.rows < PBM) tile_mainloop<true, PBM>(p, smem, acc);
    else tile_mainloop<false, PBM>(p, smem, acc);
    tile_epilogue(p, acc);
}
__device__ __forceinline__ void fp8_gemm_tile_mfma8(const TileTask& p, unsigned char* smem) {
    f32x4 acc[PTM][PTN];
    if (p.rows < PBM) tile_mainloop_mfma8<true>(p, smem, acc);
    else tile_mainloop_mfma8<false>(p, smem, acc);
    tile_epilogue(p, acc);
}

__device__ __forceinline__ TileTask resolve_tile(const FfnArgs& a, const Task& t, bool publish) {
    TileTask p;
    p.publish = publish;
    const int64_t HI = (int64_t)a.H * a.I;
    const int kbH = a.H >> 7, kbI = a.I >> 7;
    p.phase = t.phase;
    p.rows = t.rows;
    p.act = MOE_ACT_NONE;
    p.aq = t.phase == 0 ? a.xq : a.hq;
    p.sa = t.phase == 0 ? a.sx : a.sh;
    p.paired = t.phase == 0 && a.act == MOE_ACT_SWIGLU;
    if (t.phase == 0) {
        p.c0 = t.ntile * (p.paired ? PN0 : PN1);
        p.K = a.H;
        p.N = a.I;
        const int64_t srow = ((int64_t)t.expert * kbI + (p.c0 >> 7)) * kbH;
        if (p.paired) {
            p.w[0] = (const uint8_t*)a.w_gate + t.expert * HI;
            p.w[1] = (const uint8_t*)a.w_up + t.expert * HI;
            p.s[0] = a.s_gate + srow;
            p.s[1] = a.s_up + srow;
            p.bias[0] = a.b_gate ? (const uint16_t*)a.b_gate + (int64_t)t.expert * a.I : nullptr;
            p.bias[1] = a.b_up ? (const uint16_t*)a.b_up + (int64_t)t.expert * a.I : nullptr;
        } else {
            p.w[0] = p.w[1] = (const uint8_t*)a.w_up + t.expert * HI;
            p.s[0] = p.s[1] = a.s_up + srow;
            p.bias[0] = a.b_up ? (const uint16_t*)a.b_up + (int64_t)t.expert * a.I : nullptr;
            p.bias[1] = nullptr;
            p.act = a.act;
        }
        p.a_base = (const uint16_t*)a.x;
        p.gather = a.token_indices + t.row0;
        p.a_row0 = 0;
        p.c_base = (uint16_t*)a.h + (int64_t)t.row0 * a.I;
    } else {
        p.c0 = t.ntile * PN1;
        p.K = a.I;
        p.N = a.H;
        p.w[0] = p.w[1] = (const uint8_t*)a.w_down + t.expert * HI;
        const int64_t srow = ((int64_t)t.expert * kbH + (p.c0 >> 7)) * kbI;
        p.s[0] = p.s[1] = a.s_down + srow;
        p.bias[0] = a.b_down ? (const uint16_t*)a.b_down + (int64_t)t.expert * a.H : nullptr;
        p.bias[1] = nullptr;
        p.a_base = (const uint16_t*)a.h;
        p.gather = nullptr;
        p.a_row0 = t.row0;
        p.c_base = (uint16_t*)a.y + (int64_t)t.row0 * a.H;
    }
    return p;
}

__global__ __launch_bounds__(PTHREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void ffn_tiled_fp8_tile_kernel(FfnArgs a, int phase) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_list[1 + PBM];
    if (phase == 0) zero_unrouted_rows(a, 2);
    Task t;
    if (!tiled_task(a, phase, blockIdx.x, t)) return;
    const TileTask p = resolve_tile(a, t, phase == 1 && a.arrive);
    fp8_gemm_tile(p, smem);
    if (phase == 1 && a.arrive) combine_arrivals<bf16_s>(combine_args(a), t.row0, t.rows, t.ntile, p.c0, PN1, s_list);
}

__global__ __launch_bounds__(PTHREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void ffn_persistent_fp8_tile_kernel(FfnArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_task, s_ok;
    __shared__ int s_cmb[kCombineLds];
    __shared__ int s_list[1 + PBM];
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
        const TileTask p = resolve_tile(a, t, t.phase == 0 || publish_y(a));
        const long long started = trace_clock(a.task_trace);
        if (ok) fp8_gemm_tile(p, smem);
        else poison_tile(p.c_base, p.rows, p.N, p.c0, PN1, 2);
        if (a.task_trace) trace_task(a.task_trace, a.task_trace_cap, t.phase, t.expert, t.mtile, t.ntile, t.rows, started);
        if (t.phase == 0) signal_phase0_done(a.done0, t.mtile);
        else after_down_tile<bf16_s>(a, t.row0, t.rows, t.mtile, t.ntile, p.c0, PN1, s_list);
    }
    if (a.combined) combine_while_idle_narrow<bf16_s>(sweep_args(a), &s_task, s_cmb);
    queue_clock_stamp(a.wg_clock, 1);
}

// The e4m3 x e4m3 plan: one launch per projection (the intermediate rows are quantised by a pass of their own between
// the two, so the projections cannot share a queue).
__global__ __launch_bounds__(PTHREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void ffn_tiled_fp8_mfma_kernel(FfnArgs a, int phase) {
    extern __shared__ __align__(16) unsigned char smem[];
    Task t;
    if (!tiled_task(a, phase, blockIdx.x, t)) return;
    const TileTask p = resolve_tile(a, t, false);
    fp8_gemm_tile_mfma8(p, smem);
}

template <class K>
hipError_t allow_lds(K kernel) {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, PLDS);
}

}  // namespace

int fp8_tile_block_m() { return PBM; }
int fp8_tile_block_n0(int swiglu) { return swiglu ? PN0 : PN1; }
int fp8_tile_block_n1() { return PN1; }

int ffn_persistent_occupancy_fp8_tile() {
    int n = 0;
    if (allow_lds(&ffn_persistent_fp8_tile_kernel) != hipSuccess) return 1;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void*>(&ffn_persistent_fp8_tile_kernel),
                                                     PTHREADS, PLDS) != hipSuccess || n < 1)
        n = 1;
    return n;
}

hipError_t launch_ffn_fp8_tile(const FfnArgs& a, int max_mtiles, int nnt0, int nnt1, int blocks, hipStream_t st) {
    if (blocks > 0) {
        hipError_t e = allow_lds(&ffn_persistent_fp8_tile_kernel);
        if (e != hipSuccess) return e;
        ffn_persistent_fp8_tile_kernel<<<blocks, PTHREADS, PLDS, st>>>(a);
    } else {
        hipError_t e = allow_lds(&ffn_tiled_fp8_tile_kernel);
        if (e != hipSuccess) return e;
        ffn_tiled_fp8_tile_kernel<<<tiled_grid(max_mtiles, nnt0, a.groups), PTHREADS, PLDS, st>>>(a, 0);
        ffn_tiled_fp8_tile_kernel<<<tiled_grid(max_mtiles, nnt1, a.groups), PTHREADS, PLDS, st>>>(a, 1);
    }
    return hipGetLastError();
}

// x -> e4m3 rows, up projection, h -> e4m3 rows (the kept ones), down projection.
hipError_t launch_ffn_fp8_mfma(const FfnArgs& a, int S, int64_t A, int max_mtiles, int nnt0, int nnt1, hipStream_t st) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&ffn_tiled_fp8_mfma_kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, PLDS_M8);
    if (e != hipSuccess) return e;
    e = launch_quant_rows128(a.x, a.xq, a.sx, S, a.H, nullptr, st);
    if (e != hipSuccess) return e;
    ffn_tiled_fp8_mfma_kernel<<<tiled_grid(max_mtiles, nnt0, a.groups), PTHREADS, PLDS_M8, st>>>(a, 0);
    e = launch_quant_rows128(a.h, a.hq, a.sh, A, a.I, &a.q->kept_rows, st);
    if (e != hipSuccess) return e;
    ffn_tiled_fp8_mfma_kernel<<<tiled_grid(max_mtiles, nnt1, a.groups), PTHREADS, PLDS_M8, st>>>(a, 1);
    return hipGetLastError();
}

}  // namespace moe355
