// The 16-bit tiles: types, slab loops, epilogues.  Included by the layer's kernels (ffn_bf16.hip) and by the products outside the
// layer (ffn_bf16_grouped.hip).
//
// Expert FFN on bf16 MFMA: the tile GEMM "processor" of the reference, rebuilt for gfx950.
//
// Contract kept from the reference (mma.cuh:46-179, processor/tiling.cuh:273-323): C = act(A.B^T + bias)
// with A (M,K) and B (N,K) row-major, fp32 accumulation, one cast to the storage type on store, epilogue
// order add-then-activate (processor/tiling.cuh:29-38).  Everything else is designed for CDNA4:
//   * v_mfma_f32_16x16x32_bf16; the weight tile is the MFMA "A" operand and the token tile the "B" operand,
//     so each lane ends up with 4 consecutive output columns of one token row (SwiGLU pairs stay in-lane);
//   * K slabs of 64 bf16 go from global memory straight into LDS (buffer_load ... lds, no VGPR staging)
//     as 128-byte rows whose 16-byte chunks are xor-swizzled with (row >> 1) & 7: the LDS has 64 banks, a
//     ds_read_b128 is served 16 lanes at a time, and with this swizzle 16 consecutive rows of one logical
//     chunk fall into 16 distinct bank groups;
//   * two LDS stages; MFMA operand fragments are double buffered in registers;
//   * dispatch is fused into the A-tile load: phase 0 gathers token rows through token_indices[];
//   * SwiGLU pairs gate and up columns inside one wavefront (first half of its tile rows from w_gate, second
//     half from w_up), so silu(g)*u happens in registers.
// Plans: "large", 256-row blocks and 256 x 256 tiles, four wavefronts of 128 x 128; "medium", 128-row blocks and 128 x 256
// tiles, four wavefronts of 128 x 64; both with the slab loop ordered by hand (gemm_tile_ring) and an epilogue staged
// through LDS, for operands below 4 GiB, chosen by bf16_tile.  "Small": 128 x 128 tiles, four wavefronts of 64 x 64,
// compiler-scheduled loop (mainloop_generic), general epilogue; takes everything else.
#pragma once

#include <type_traits>

#include "ffn_common.hpp"
#include "act_deriv.hpp"
#include "product_choice.hpp"
#include "two_launches.hpp"

namespace moe355 {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void gbl_void;

constexpr int kBK = 64;               // bf16 elements of K per slab = one 128-byte LDS row
constexpr int kRowBytes = kBK * 2;

// F16: operands and results are IEEE binary16 (torch_dtype 3) instead of bfloat16; same tile, same loops, the other
// MFMA instruction and the other conversions.
// TRA, TRB: the token / weight operand is stored with k as its slow index (hand-ordered tiles only; ring_load_one).
template <int BM_, int BN_, int WM_, int WN_, int NS_, bool F16_ = false, bool TRA_ = false, bool TRB_ = false>
struct Tile {
    static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, NS = NS_;
    static constexpr bool F16 = F16_, TRA = TRA_, TRB = TRB_;
    static constexpr bool PIECES = false;         // fp32 operands as three bf16 pieces (ffn_f32_pieces.hip)
    static constexpr int THREADS = WM * WN * kWave;
    static constexpr int TM = BM / WM / 16;       // 16x16 MFMA tiles per wavefront along tokens
    static constexpr int TN = BN / WN / 16;       // ... along weight rows
    static constexpr int ROWS_PER_PASS = THREADS / 8;
    static constexpr int RA = BM / ROWS_PER_PASS; // 16-byte loads per thread per slab, token tile
    static constexpr int RB = BN / ROWS_PER_PASS; // ... weight tile
    static constexpr int STAGE_BYTES = (BM + BN) * kRowBytes;
    // four wavefronts of 128 x 128 outputs: this tile runs the hand-ordered slab loop (gemm_tile_ring)
    static constexpr bool RING = BM == 256 && BN == 256 && WM == 2 && WN == 2;
    // four wavefronts of 128 x 64 outputs, side by side (128 x 256) or two by two (256 x 128): the same loop with
    // half the weight fragments per wavefront
    static constexpr bool HALF = TM == 8 && TN == 4 && WM * WN == 4;
    static constexpr bool HAND = RING || HALF;
    static constexpr int WB = BN / WN;            // weight rows per wavefront
    // behind the stages: where the four wavefronts of a hand-ordered tile turn 16 rows of results at a time into
    // row-major order (row pitch: the wavefront's columns in bytes + 16)
    static constexpr int STAGING_BYTES = HAND ? 4 * 16 * (TN * 32 + 16) : 0;
    static constexpr int LDS_BYTES = NS * STAGE_BYTES + STAGING_BYTES;
    static_assert(TM >= 2 && TM % 2 == 0 && TN >= 2 && TN % 2 == 0, "a wavefront's tile is split in token halves; SwiGLU pairs weight-row halves");
    static_assert(RA >= 1 && RB >= 1, "tile too small for the workgroup");
    static_assert(NS == 2, "two LDS stages");
    static_assert(HAND || !(TRA || TRB), "operands with k as their slow index: the hand-ordered tiles");
    static_assert(TRB || !TRA, "slab orders exist for the weights alone or both operands");
};

// What one task needs, resolved to pointers.
struct TaskPtrs {
    const uint16_t* a_base;      // phase 0: x; phase 1: h
    const int32_t* gather;       // phase 0: token_indices + row0; phase 1: null
    int64_t a_row0;              // phase 1: first row of h
    int a_ld;                    // K
    const uint16_t* b0;          // weight matrix of this expert (w_up or w_down)
    const uint16_t* b1;          // SwiGLU: w_gate of this expert, else null
    int b_ld;                    // elements between weight rows (K unless the operand is a window of a wider matrix)
    const uint16_t* bias0;
    const uint16_t* bias1;
    uint16_t* c_base;            // h or y, first row of the block
    int N;                       // output columns (I for phase 0, H for phase 1)
    int K;
    int rows;
    int n0;                      // first output column of this tile
    int act;                     // epilogue
    bool swiglu;
    bool publish;                // the rows will be read by other workgroups of the same launch
    uint32_t a_extent, b_extent; // bytes of the token operand (from a_base) and of one weight matrix (from b0 / b1)
    // A task that is one of `kparts` partial sums of its tile over the contraction dimension (null part: a whole tile):
    float* part;                 // the tile's partial-sum buffers, kparts x (block rows x block columns) fp32
    int32_t* part_cnt;           // parts of the tile stored so far
    int kparts, kpart;
    bool poison;                 // such a task whose rows never became ready: its part is NaN
    // The data gradient of the down projection with the activation's derivative in its epilogue (grouped kernel only;
    // deriv 0: an ordinary task): the tile's sums are dh, and what is stored is dh * act'(u) (and, for SwiGLU, the gate's
    // share beside it) from the saved projections u (and g), which have the output's shape.
    int deriv;                   // 0, or 1 + the layer's hidden_act
    const uint16_t* aux0;        // u rows, first row of the block
    const uint16_t* aux1;        // g rows (SwiGLU), else null
    uint16_t* c1_base;           // dg rows (SwiGLU), else null
};

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// Two fp32 values rounded to the tile's 16-bit storage type (nearest even), and one stored value widened.
template <class T>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    if constexpr (T::F16) {
        typedef float f32x2_t __attribute__((ext_vector_type(2)));
        typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
        const f32x2_t v = {lo, hi};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2_t));
    } else {
        return pack2_bf16(lo, hi);
    }
}
template <class T>
__device__ __forceinline__ float widen1(uint16_t v) {
    if constexpr (T::F16) return (float)__builtin_bit_cast(_Float16, v);
    else return bf16_bits_to_f32(v);
}

// 8 bytes of output; rows that another workgroup of the same launch will read are published (ffn_common.hpp).
__device__ __forceinline__ void store8(uint16_t* p, uint32_t lo, uint32_t hi, bool publish) {
    if (publish) {
        publish8(p, lo, hi);
    } else {
        u32x2 o = {lo, hi};
        *reinterpret_cast<u32x2*>(p) = o;
    }
}

// PARTIAL: the row block holds fewer than BM rows; 16-row MFMA sub-tiles that lie entirely in the padding are
// skipped (their LDS reads too).  A separate instantiation keeps the full-tile loop free of branches.
//
// Loop structure.  A 64-wide slab is consumed in four units (k half s, token half h) of HM x TN MFMAs; the
// fragments of the next unit are read from LDS under the MFMAs of the current one.  The one barrier per slab sits
// before the last unit: by then every wavefront has read all of the slab's fragments, so the barrier both frees
// this stage for the loads of slab kt+2 (issued right behind it) and publishes slab kt+1, whose first fragments
// are read under the last unit's MFMAs.  The first and the last two slabs are peeled off so that the steady-state
// loop is one basic block, which is what lets the scheduling hints hold.
template <class T, bool PARTIAL>
__device__ __forceinline__ void mainloop_generic(const TaskPtrs& p, unsigned char* smem, f32x4 (&acc)[T::TM][T::TN]) {
    constexpr int BM = T::BM, BN = T::BN, TM = T::TM, TN = T::TN, HM = TM / 2;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / T::WN, wn = wave % T::WN;
    const int prow = tid >> 3;
    const int chunk = (tid & 7) ^ ((prow >> 1) & 7);   // LDS slot (row, c) holds global chunk c ^ ((row >> 1) & 7)

    // ---- per-thread source rows ----
    const uint16_t* a_src[T::RA];
    const uint16_t* b_src[T::RB];
#pragma unroll
    for (int i = 0; i < T::RA; ++i) {
        int r = prow + i * T::ROWS_PER_PASS;
        if (r >= p.rows) r = 0;                                   // padding rows re-read row 0; never stored
        const int64_t src_row = p.gather ? (int64_t)p.gather[r] : p.a_row0 + r;
        a_src[i] = p.a_base + src_row * p.a_ld + chunk * 8;
    }
#pragma unroll
    for (int i = 0; i < T::RB; ++i) {
        const int j = prow + i * T::ROWS_PER_PASS;                // row of the weight tile
        const uint16_t* base = p.b0;
        int col;
        if (p.swiglu) {
            constexpr int WCOLS = BN / T::WN;                     // tile rows owned by one wavefront column
            const int w = j / WCOLS, jj = j % WCOLS;
            const int half = jj / (WCOLS / 2);
            col = p.n0 + w * (WCOLS / 2) + (jj % (WCOLS / 2));
            base = half ? p.b0 : p.b1;                            // first half gate, second half up
        } else {
            col = p.n0 + j;
        }
        if (col >= p.N) col = p.N - 1;                            // ragged last tile; never stored
        b_src[i] = base + (int64_t)col * p.b_ld + chunk * 8;
    }

#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.0f;

    // One global_load_lds_dwordx4 per 8 rows and wavefront writes 1 KiB of consecutive LDS: lane l lands in
    // row (l >> 3), chunk slot (l & 7); the swizzle is applied on the global side (see `chunk`).
    const int wrow = __builtin_amdgcn_readfirstlane(prow & ~7);
    const int KT = p.K / kBK;
    auto issue = [&](int kt) {
        unsigned char* sa = smem + (kt & 1) * T::STAGE_BYTES;
        unsigned char* sb = sa + BM * kRowBytes;
        const int koff = kt * kBK;
#pragma unroll
        for (int i = 0; i < T::RA; ++i)
            __builtin_amdgcn_global_load_lds((gbl_void*)(a_src[i] + koff),
                                             (lds_void*)(sa + (wrow + i * T::ROWS_PER_PASS) * kRowBytes), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < T::RB; ++i)
            __builtin_amdgcn_global_load_lds((gbl_void*)(b_src[i] + koff),
                                             (lds_void*)(sb + (wrow + i * T::ROWS_PER_PASS) * kRowBytes), 16, 0, 0);
    };
    __syncthreads();                        // the previous task may still be reading the stages
    issue(0);
    if (KT > 1) issue(1);

    const int frow = lane & 15, fk = lane >> 4;
    const int sw = (frow >> 1) & 7;
    // 16-row sub-tiles of this wavefront that contain at least one real row (wavefront-uniform)
    const int ta = PARTIAL ? min(TM, max(0, (p.rows - wm * 16 * TM + 15) >> 4)) : TM;
    const int a_base = (wm * 16 * TM + frow) * kRowBytes;
    const int b_base = BM * kRowBytes + (wn * 16 * TN + frow) * kRowBytes;

    bf16x8 af[2][HM], bfr[2][TN];
    auto read_a = [&](const unsigned char* st, int s, int h, int buf) {
        const int c = ((s * 4 + fk) ^ sw) << 4;
#pragma unroll
        for (int i = 0; i < HM; ++i)
            if (!PARTIAL || h * HM + i < ta)
                af[buf][i] = *reinterpret_cast<const bf16x8*>(st + a_base + (h * HM + i) * 16 * kRowBytes + c);
    };
    auto read_b = [&](const unsigned char* st, int s, int buf) {
        const int c = ((s * 4 + fk) ^ sw) << 4;
#pragma unroll
        for (int j = 0; j < TN; ++j) bfr[buf][j] = *reinterpret_cast<const bf16x8*>(st + b_base + j * 16 * kRowBytes + c);
    };
    auto mfmas = [&](int h, int abuf, int bbuf) {
#pragma unroll
        for (int i = 0; i < HM; ++i) {
            if (PARTIAL && h * HM + i >= ta) continue;
#pragma unroll
            for (int j = 0; j < TN; ++j)
                acc[h * HM + i][j] =
                    T::F16 ? __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, bfr[bbuf][j]),
                                                                      __builtin_bit_cast(f16x8, af[abuf][i]), acc[h * HM + i][j], 0, 0, 0)
                           : __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[bbuf][j], af[abuf][i], acc[h * HM + i][j], 0, 0, 0);
        }
    };
    // instruction order inside a unit: behind every second MFMA one LDS read and (last unit) one global load
    auto hints = [&](auto nds_c, auto nvm_c) {
        constexpr int nds = decltype(nds_c)::value, nvm = decltype(nvm_c)::value;
        if (PARTIAL) return;
        constexpr int npair = nds > nvm ? nds : nvm;
        constexpr int NM = HM * TN;
#pragma unroll
        for (int n = 0; n < npair; ++n) {
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
            if (n < nds) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            if (n < nvm) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        }
        if (NM > 2 * npair) __builtin_amdgcn_sched_group_barrier(0x008, NM - 2 * npair, 0);
    };
    constexpr int NLOADS = T::RA + T::RB;
    typedef std::integral_constant<int, 0> Zero;

    // slab 0 has landed when at most the loads of slab 1 are outstanding (loads return in issue order)
    if (KT > 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NLOADS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    read_a(smem, 0, 0, 0);
    read_b(smem, 0, 0);
    auto slab = [&](auto more_c, auto pre2_c, int kt) {
        constexpr bool MORE = decltype(more_c)::value, PRE2 = decltype(pre2_c)::value;
        const unsigned char* st = smem + (kt & 1) * T::STAGE_BYTES;
        const unsigned char* sn = smem + ((kt + 1) & 1) * T::STAGE_BYTES;
        read_a(st, 0, 1, 1);
        mfmas(0, 0, 0);
        hints(std::integral_constant<int, HM>{}, Zero{});
        read_a(st, 1, 0, 0);
        read_b(st, 1, 1);
        mfmas(1, 1, 0);
        hints(std::integral_constant<int, HM + TN>{}, Zero{});
        read_a(st, 1, 1, 1);
        mfmas(0, 0, 1);
        hints(std::integral_constant<int, HM>{}, Zero{});
        // every fragment of slab kt is in registers; this wavefront's share of slab kt+1 has landed
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __syncthreads();
        if (MORE) {
            read_a(sn, 0, 0, 0);
            read_b(sn, 0, 0);
        }
        if (PRE2) issue(kt + 2);
        mfmas(1, 1, 1);
        hints(std::integral_constant<int, MORE ? HM + TN : 0>{}, std::integral_constant<int, PRE2 ? NLOADS : 0>{});
    };
    int kt = 0;
    for (; kt < KT - 2; ++kt) slab(std::true_type{}, std::true_type{}, kt);
    if (KT > 1) {
        slab(std::true_type{}, std::false_type{}, kt);
        ++kt;
    }
    slab(std::false_type{}, std::false_type{}, kt);
}

// acc[i][j][r]: token row = wm*16*TM + i*16 + (lane & 15); weight row inside the 16-wide MFMA tile = 4*(lane >> 4) + r.
// MODE: 0 none / ReLU, 2 GELU (erf form), 3 SwiGLU.  The choice is made once per tile so that the unrolled store loop
// does not branch around the (large) GELU code for every element.
template <class T, int MODE>
__device__ __forceinline__ void epilogue_impl(const TaskPtrs& p, f32x4 (&acc)[T::TM][T::TN]) {
    constexpr int TM = T::TM, TN = T::TN;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave / T::WN, wn = wave % T::WN;
    const int frow = lane & 15, fk = lane >> 4;
    // MODE 0: u below the floor becomes the floor.  Written as a compare and select, not as fmaxf: a max returns its
    // other operand for a NaN, and a NaN must stay a NaN (the reference's __hfma_relu propagates it too, processor/tiling.cuh:45,54)
    const float relu_floor = p.act == MOE_ACT_RELU ? 0.0f : -INFINITY;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int m = wm * 16 * TM + i * 16 + frow;
        if (m >= p.rows) continue;
        uint16_t* crow = p.c_base + (int64_t)m * p.N;
        if constexpr (MODE == 3) {
#pragma unroll
            for (int j = 0; j < TN / 2; ++j) {
                const int col = p.n0 + wn * 8 * TN + j * 16 + 4 * fk;
                if (col >= p.N) continue;
                float v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float g = acc[i][j][r], u = acc[i][j + TN / 2][r];
                    if (p.bias1) g = g + widen1<T>(p.bias1[col + r]);
                    if (p.bias0) u = u + widen1<T>(p.bias0[col + r]);
                    v[r] = silu16(g) * u;
                }
                store8(crow + col, pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3]), p.publish);
            }
        } else {
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int col = p.n0 + wn * 16 * TN + j * 16 + 4 * fk;
                if (col >= p.N) continue;
                float v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float u = acc[i][j][r];
                    if (p.bias0) u = u + widen1<T>(p.bias0[col + r]);
                    v[r] = MODE == 2 ? gelu16(u) : (u < relu_floor ? relu_floor : u);
                }
                store8(crow + col, pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3]), p.publish);
            }
        }
    }
}

template <class T>
__device__ __forceinline__ void epilogue(const TaskPtrs& p, f32x4 (&acc)[T::TM][T::TN]) {
    if (p.swiglu) epilogue_impl<T, 3>(p, acc);
    else if (p.act == MOE_ACT_GELU) epilogue_impl<T, 2>(p, acc);
    else epilogue_impl<T, 0>(p, acc);
}

// The epilogue of the hand-ordered tiles, staged through LDS.
//
// In the accumulator layout the 16 lanes that are neighbours in the wavefront hold 16 different rows, so a store
// straight from the registers writes 64 separate 8-byte pieces per instruction.  Each wavefront therefore writes its
// bf16 results, 16 rows at a time, into its own piece of LDS behind the slab stages and reads them back row-major:
// 16 bytes per lane, a whole row of the wavefront's columns per 16 (8 for SwiGLU) neighbouring lanes, four (eight)
// rows per store instruction.  No barrier is involved (same wavefront, LDS operations complete in order), and the
// slab stages stay free: the loads of the workgroup's next task may already be landing in them.  The row pitch is
// padded by 16 bytes, which puts the 8-byte writes of 32 neighbouring lanes on distinct banks.  The bias values of
// this lane's columns are loaded once (or are -0.0f, the neutral element of the addition), so the element loop has
// no branch.
// A store of more than 8 bytes reads its data registers over the cycles behind its issue, and an instruction that
// writes one of them must keep two wait states' distance.  The compiler sees to that for the stores it emits, not for one
// inside an asm statement -- it may well put the next value into the same registers right behind it -- so the statement
// brings the wait states along.
#define MOE_STORE16_AGENT "global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1"
__device__ __forceinline__ void store16(uint16_t* p, u32x4 v, bool publish) {
    if (publish) asm volatile(MOE_STORE16_AGENT ::"v"(p), "v"(v) : "memory");   // agent scope, as publish8
    else *reinterpret_cast<u32x4*>(p) = v;
}

struct NoHook {
    __device__ __forceinline__ void operator()(int) const {}
};
// The epilogue of a tile that was computed as KP partial sums (partial_tile_arrive): `base` is this lane's place in the
// partial-sum buffers of the tile (two parts: in the other part's buffer; four parts: in the buffer of part 0).
struct WholeTile {
    static constexpr int KP = 1;
};
template <int KP_>
struct SummedTile {
    static constexpr int KP = KP_;
    const float* base;
};

// `between(i)` runs in front of row group i (i = 0..7): the queue kernel issues the next task's first loads there, a
// few at a time, so that they leave the compute unit under the epilogue's arithmetic instead of in front of it.
// DERIV: what leaves the staging area is not stored as it is (dh, rounded to 16 bits as a stored data gradient would be)
// but multiplied by the activation's derivative at the saved projections (TaskPtrs::deriv): a row segment's 8 values
// meet the 8 values of u (and g) of the same rows and columns, loaded at the top of the row group.
template <class T, int MODE, class Hook, class Parts = WholeTile, bool DERIV = false>
__device__ __forceinline__ void epilogue_full_n_impl(const TaskPtrs& p, unsigned char* smem, f32x4 (&acc)[T::TM][T::TN], const Hook& between,
                                                     const Parts& parts = Parts()) {
    static_assert(Parts::KP == 1 || MODE == 0, "partial sums: the down projection only");
    static_assert(!DERIV || (MODE == 0 && Parts::KP == 1), "the derivative follows a plain product");

    static_assert(T::HAND, "four wavefronts of 128 or 64 columns");
    constexpr int NJ = MODE == 3 ? T::TN / 2 : T::TN;   // groups of 16 output columns per wavefront
    constexpr int ROW_BYTES = NJ * 32, PITCH = ROW_BYTES + 16;
    constexpr int LANES_PER_ROW = ROW_BYTES / 16, ROWS_PER_PASS = 64 / LANES_PER_ROW;
    static_assert(T::WM * T::WN * 16 * PITCH <= T::STAGING_BYTES, "the staging pieces of the wavefronts fit behind the slab stages");
    // Everything below is derived from a thread id the compiler cannot see through: otherwise it computes these
    // addresses before the slab loop, finds no register to keep them in, and reloads them from scratch memory
    // between the stores (each reload then waits for the store before it).
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / T::WN, wn = wave % T::WN;
    const int frow = lane & 15, fk = lane >> 4;
    const int col0 = p.n0 + wn * 16 * NJ;        // first output column of this wavefront
    // Columns behind the last one: N is a multiple of 64, so each of the wavefront's 64 columns (32 with SwiGLU on the smaller
    // tile) exist together or not at all, and what the masks need is the same in every lane.  (Per lane -- a minimum in every
    // bias address, a compare in rows_left -- they cost the layers that need none 1 %: 16 experts of 2048 x 2048, 512 rows each, 215.1
    // against 212.7 us without masks; as they stand 217.4 against 217.0, another card.)
    const int col_lo = col0 < p.N ? col0 : 0, col_hi = col0 + 64 < p.N ? col0 + 64 : 0;
    float b0[NJ][4], b1[NJ][4];
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) b0[j][r] = b1[j][r] = -0.0f;
    if (p.bias0) {
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) b0[j][r] = widen1<T>(p.bias0[(j < 4 ? col_lo : col_hi) + 16 * (j % 4) + 4 * fk + r]);
    }
    if (MODE == 3 && p.bias1) {
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) b1[j][r] = widen1<T>(p.bias1[(j < 4 ? col_lo : col_hi) + 16 * (j % 4) + 4 * fk + r]);
    }
    // MODE 0: u below the floor becomes the floor.  Written as a compare and select, not as fmaxf: a max returns its
    // other operand for a NaN, and a NaN must stay a NaN (the reference's __hfma_relu propagates it too, processor/tiling.cuh:45,54)
    const float relu_floor = p.act == MOE_ACT_RELU ? 0.0f : -INFINITY;
    unsigned char* stage = smem + T::NS * T::STAGE_BYTES + wave * (16 * PITCH);
    unsigned char* wr = stage + frow * PITCH + fk * 8;
    const int rd_row = lane / LANES_PER_ROW, rd_chunk = lane % LANES_PER_ROW;
    const unsigned char* rd = stage + rd_row * PITCH + rd_chunk * 16;
    // this lane stores row r0 + rd_row when r0 < rows_left; none if its eight columns lie behind the last one
    int rows_left = (col0 < p.N ? p.rows - wm * 16 * T::TM : 0) - rd_row;
    if (NJ == 8 && col0 + 64 >= p.N && rd_chunk >= 8) rows_left = 0;
    const uint32_t lane_off = (uint32_t)(rd_row * p.N + col0 + rd_chunk * 8);   // elements from the uniform row pointer
    const bool publish = p.publish;
    constexpr int NQ = 16 / ROWS_PER_PASS;
    // (DERIV) the saved projections, requested kAhead row groups in front of the one that uses them: nothing else in flight on the
    // SIMD hides their way from memory.  Against requests at the top of their own group, a SwiGLU data gradient on the 128 x 256
    // tile: 16 experts of 2048 x 2048, 512 rows each 148 -> 137 us; of 2048 x 1408, 750 rows 131 -> 119; 16 of 1152 x 1920, 175 rows 33.8 -> 31.6.
    constexpr int kAhead = T::RING ? 3 : 2;
    u32x4 saved_u[DERIV ? kAhead + 1 : 1][NQ], saved_g[DERIV ? kAhead + 1 : 1][NQ];
    auto saved_rows = [&](int i) {
        if (i >= T::TM) return;
        const int64_t group = (int64_t)(wm * 16 * T::TM + i * 16) * p.N;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            u32x4 &u = saved_u[i % (kAhead + 1)][q], &g = saved_g[i % (kAhead + 1)][q];
            u = g = u32x4{0u, 0u, 0u, 0u};
            if (i * 16 + q * ROWS_PER_PASS < rows_left) {
                const int64_t at = group + (int64_t)(q * ROWS_PER_PASS) * p.N + lane_off;
                u = *reinterpret_cast<const u32x4*>(p.aux0 + at);
                if (p.deriv == 1 + MOE_ACT_SWIGLU) g = *reinterpret_cast<const u32x4*>(p.aux1 + at);
            }
        }
    };
    if constexpr (DERIV) {
#pragma unroll
        for (int i = 0; i < kAhead; ++i) saved_rows(i);
    }
#pragma unroll
    for (int i = 0; i < T::TM; ++i) {
        between(i);
        if constexpr (DERIV) saved_rows(i + kAhead);
        // Partial sums: the row group's sums of the other parts come back from memory (written through by their tasks,
        // read past this XCD's L2) and are added here -- two parts: own registers + the other part, which is the same
        // in either order; four parts: all four as stored, in the order of the parts, whichever of them runs this.
        f32x4 whole[Parts::KP == 1 ? 1 : NJ];
        if constexpr (Parts::KP == 2) {
#pragma unroll
            for (int j = 0; j < NJ; ++j)
                asm volatile("global_load_dwordx4 %0, %1, off sc1" : "=v"(whole[j]) : "v"(parts.base + (i * NJ + j) * 256) : "memory");
#pragma unroll
            for (int j = 0; j < NJ; ++j) asm volatile("s_waitcnt vmcnt(0)" : "+v"(whole[j])::"memory");
#pragma unroll
            for (int j = 0; j < NJ; ++j) whole[j] = acc[i][j] + whole[j];
        } else if constexpr (Parts::KP == 4) {
            constexpr size_t kPartFloats = (size_t)T::BM * T::BN;
#pragma unroll
            for (int j0 = 0; j0 < NJ; j0 += 4) {
                f32x4 v[4][4];
#pragma unroll
                for (int k = 0; k < 4; ++k)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        asm volatile("global_load_dwordx4 %0, %1, off sc1" : "=v"(v[k][j]) : "v"(parts.base + k * kPartFloats + (i * NJ + j0 + j) * 256) : "memory");
#pragma unroll
                for (int k = 0; k < 4; ++k)
#pragma unroll
                    for (int j = 0; j < 4; ++j) asm volatile("s_waitcnt vmcnt(0)" : "+v"(v[k][j])::"memory");
#pragma unroll
                for (int j = 0; j < 4; ++j) whole[j0 + j] = ((v[0][j] + v[1][j]) + v[2][j]) + v[3][j];
            }
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if constexpr (MODE == 3) {
                    const float g = acc[i][j][r] + b1[j][r], u = acc[i][j + NJ][r] + b0[j][r];
                    v[r] = silu16(g) * u;
                } else {
                    float sum;
                    if constexpr (Parts::KP == 1) sum = acc[i][j][r]; else sum = whole[j][r];
                    const float u = sum + b0[j][r];
                    v[r] = MODE == 2 ? gelu16(u) : (u < relu_floor ? relu_floor : u);
                }
            }
            u32x2 o = {pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
            *reinterpret_cast<u32x2*>(wr + j * 32) = o;
        }
        u32x4 v[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) v[q] = *reinterpret_cast<const u32x4*>(rd + q * ROWS_PER_PASS * PITCH);
        uint16_t* rows0 = p.c_base + (int64_t)(wm * 16 * T::TM + i * 16) * p.N;   // uniform
        if constexpr (DERIV) {
            const int64_t group = (int64_t)(wm * 16 * T::TM + i * 16) * p.N;
            const bool gated = p.deriv == 1 + MOE_ACT_SWIGLU;
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                if (i * 16 + q * ROWS_PER_PASS >= rows_left) continue;
                const int64_t at = group + (int64_t)(q * ROWS_PER_PASS) * p.N + lane_off;
                u32x4 o0, o1 = {0u, 0u, 0u, 0u};
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const float d0 = widen1<T>((uint16_t)(v[q][w] & 0xFFFFu)), d1 = widen1<T>((uint16_t)(v[q][w] >> 16));
                    const u32x4 uu = saved_u[i % (kAhead + 1)][q], gg = saved_g[i % (kAhead + 1)][q];
                    const float u0 = widen1<T>((uint16_t)(uu[w] & 0xFFFFu)), u1 = widen1<T>((uint16_t)(uu[w] >> 16));
                    float a0, a1, b0v = 0.0f, b1v = 0.0f;
                    if (gated) {
                        const float g0 = widen1<T>((uint16_t)(gg[w] & 0xFFFFu)), g1 = widen1<T>((uint16_t)(gg[w] >> 16));
                        dswiglu16(d0, u0, g0, a0, b0v);
                        dswiglu16(d1, u1, g1, a1, b1v);
                    } else if (p.deriv == 1 + MOE_ACT_GELU) {
                        a0 = dgelu16(d0, u0);
                        a1 = dgelu16(d1, u1);
                    } else {
                        a0 = drelu16(d0, u0);
                        a1 = drelu16(d1, u1);
                    }
                    o0[w] = pack2<T>(a0, a1);
                    o1[w] = pack2<T>(b0v, b1v);
                }
                store16(p.c_base + at, o0, false);
                if (gated) store16(p.c1_base + at, o1, false);
            }
            continue;
        }
        if (publish) {
#pragma unroll
            for (int q = 0; q < NQ; ++q)
                if (i * 16 + q * ROWS_PER_PASS < rows_left)
                    store16(rows0 + (int64_t)(q * ROWS_PER_PASS) * p.N + lane_off, v[q], true);
        } else {
#pragma unroll
            for (int q = 0; q < NQ; ++q)
                if (i * 16 + q * ROWS_PER_PASS < rows_left)
                    store16(rows0 + (int64_t)(q * ROWS_PER_PASS) * p.N + lane_off, v[q], false);
        }
    }
}

template <class T, class Hook = NoHook>
__device__ __forceinline__ void epilogue_full_n(const TaskPtrs& p, unsigned char* smem, f32x4 (&acc)[T::TM][T::TN], const Hook& between = Hook()) {
    if (p.swiglu) epilogue_full_n_impl<T, 3>(p, smem, acc, between);
    else if (p.act == MOE_ACT_GELU) epilogue_full_n_impl<T, 2>(p, smem, acc, between);
    else epilogue_full_n_impl<T, 0>(p, smem, acc, between);
}

// What the loads of one task of the hand-ordered tile need; computed once per task (ring_prepare).
struct RingLoads {
    unsigned voff_a[8], voff_b[8];   // byte offsets of this thread's eight token rows / weight rows (row + 16-byte chunk)
    const void* base_a;              // wavefront-uniform operand bases
    const void* base_b0;
    const void* base_b1;
    uint32_t a_extent, b_extent;
    uint32_t a_slab, b_slab;         // TRA, TRB: bytes of a slab's 64 k
    uint32_t piece_slabs, piece_recip;   // PIECES: slabs of one piece, and 2^32 over it, rounded up
    int KT;                          // slabs of 64, >= 1
    int wrow;                        // first of the eight consecutive stage rows this wavefront's loads fill per pass
};

// Operands with k as their slow index (TRA, TRB).  A slab is 64 rows of k, each as long as the tile is wide (W elements), and goes
// into the stage as it lies in memory.  What turns it round is the fragment read: ds_read_b64_tr_b16 gives lane i of sixteen the
// i-th column of the 4 x 16 block whose rows its groups of four lanes address, so two of them make the eight k of a lane's
// operand, the same k in the same places as from an operand stored the other way: same bits.  (Turning the operand in registers on
// its way to LDS, 128 x 128 tiles on two workgroups a compute unit: ProdTile, ffn_bf16_grouped.hip.)
// A wavefront's read meets rows of k that lie a multiple of 256 bytes apart, eight at a time; the 32-byte pieces of a row are
// therefore permuted within every eight, by turned_swizzle, on the global side of the loads and in the addresses of the reads.
__device__ __forceinline__ int turned_swizzle(int k) { return (k & 3) | ((k >> 1) & 4); }
// Byte offsets of this thread's loads of a slab, from its first row of k on: load n of a wavefront fills 1 KiB of the stage.
template <int W>
__device__ __forceinline__ void turned_offsets(int ld, int tid, unsigned (&voff)[8]) {
    constexpr int PITCH = W * 2;
#pragma unroll
    for (int n = 0; n < W / 32; ++n) {
        const int at = n * 4096 + tid * 16, k = at / PITCH, piece = at % PITCH / 32;
        voff[n] = (unsigned)(k * ld * 2 + (piece ^ turned_swizzle(k)) * 32 + (at & 16));
    }
}
// This lane's place in the stage for its fragment `f` (sixteen columns) of k 0..31; the second four of its k lie 4 rows on.
template <int W>
__device__ __forceinline__ unsigned turned_fragment(int f, int lane) {
    const int k = 8 * (lane >> 4) + ((lane >> 2) & 3);
    return (unsigned)(k * (W * 2) + (f ^ turned_swizzle(k)) * 32 + (lane & 3) * 8);
}

// The part of a task's load state that needs no memory access: weight-row offsets, bases, extents.
template <class T>
__device__ __forceinline__ RingLoads ring_prepare_weights(const TaskPtrs& p) {
    static_assert(T::HAND && T::ROWS_PER_PASS == 32, "four wavefronts of 128 x 128 or 128 x 64");
    // a thread id the compiler cannot see through: what is derived from it is computed here, not once at the top of
    // the kernel and then kept (and spilled) across the slab loop
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int prow = tid >> 3;
    const int chunk = (tid & 7) ^ ((prow >> 1) & 7);
    RingLoads L;
#pragma unroll
    for (int n = 0; n < 8; ++n) L.voff_a[n] = L.voff_b[n] = p.a_extent;
    if constexpr (T::TRB) turned_offsets<T::BN>(p.b_ld, tid, L.voff_b);
#pragma unroll
    for (int n = 0; n < (T::TRB ? 0 : T::RB); ++n) {
        // SwiGLU: a wavefront's weight rows are the gate rows of its output columns followed by their up rows
        const int j = prow + n * T::ROWS_PER_PASS;
        const int col = p.swiglu ? p.n0 + (j / T::WB) * (T::WB / 2) + (j % (T::WB / 2)) : p.n0 + j;
        // (columns behind the last one of a ragged tile lie behind the end of the matrix, hence of the buffer)
        L.voff_b[n] = (unsigned)(((int64_t)col * p.b_ld + chunk * 8) * 2);
    }
    auto uniform = [](const void* q) {          // the bases are the same in every lane; say so, or each load loops over lanes
        const uint64_t v = (uint64_t)q;
        // readfirstlane returns int: go through uint32_t, or a low half with bit 31 set sign-extends over the high half
        const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
        const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
        return (const void*)(((uint64_t)hi << 32) | (uint64_t)lo);
    };
    L.base_a = uniform(p.a_base);
    L.base_b0 = uniform(p.b0);
    L.base_b1 = uniform(p.swiglu ? p.b1 : p.b0);
    L.a_extent = p.a_extent;
    L.b_extent = p.b_extent;
    L.a_slab = T::TRA ? (uint32_t)p.a_ld * kRowBytes : 0u;
    L.b_slab = T::TRB ? (uint32_t)p.b_ld * kRowBytes : 0u;
    L.KT = p.K / kBK;
    L.piece_slabs = T::PIECES ? (uint32_t)L.KT / 6u : 0u;
    L.piece_recip = T::PIECES ? 0xFFFFFFFFu / L.piece_slabs + 1u : 0u;
    L.wrow = __builtin_amdgcn_readfirstlane(prow & ~7);
    return L;
}

// The token-row offsets: phase 0 gathers the row numbers through token_indices[] (eight loads per thread).
template <class T>
__device__ __forceinline__ void ring_prepare_tokens(const TaskPtrs& p, RingLoads& L) {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int prow = tid >> 3;
    const int chunk = (tid & 7) ^ ((prow >> 1) & 7);
    if constexpr (T::TRA) {
        turned_offsets<T::BM>(p.a_ld, tid, L.voff_a);
        return;
    }
#pragma unroll
    for (int n = 0; n < T::RA; ++n) {
        // Padding rows are never stored.  Their loads are aimed behind the end of the buffer, which the hardware
        // answers with zeros without touching memory: MFMAs on zeros draw less of the power budget than MFMAs on a
        // copy of real rows.
        const int r0 = prow + n * T::ROWS_PER_PASS, r = max(min(r0, p.rows - 1), 0);
        const int64_t src_row = p.gather ? (int64_t)p.gather[r] : p.a_row0 + r;
        L.voff_a[n] = r0 < p.rows ? (unsigned)((src_row * p.a_ld + chunk * 8) * 2) : p.a_extent;
    }
}

template <class T>
__device__ __forceinline__ RingLoads ring_prepare(const TaskPtrs& p) {
    RingLoads L = ring_prepare_weights<T>(p);
    ring_prepare_tokens<T>(p, L);
    return L;
}

// fp32 operands as three bf16 pieces, a row one piece behind the other (ffn_f32_pieces.hip): the contraction runs over six pairs of
// pieces, the smallest products first.
constexpr uint32_t kPieceA = 2u | 0u << 2 | 1u << 4 | 1u << 6 | 0u << 8 | 0u << 10, kPieceB = 0u | 2u << 2 | 1u << 4 | 0u << 6 | 1u << 8 | 0u << 10;
__device__ __forceinline__ int piece_offset(const RingLoads& L, int slab, uint32_t pieces) {
    const uint32_t pair = __umulhi((uint32_t)slab, L.piece_recip);      // slab / piece_slabs (slab < 7 * 2^10)
    return (int)((((pieces >> (2 * pair)) & 3u) * L.piece_slabs + ((uint32_t)slab - pair * L.piece_slabs)) * kRowBytes);
}

// Load n of slab `slab` of a task: n < RA token rows, else weight rows; the weight rows of pass m come from w_gate when
// they lie in the first half of a wavefront's weight rows.  Raw buffers (stride 0) that end where the operand ends.  Slabs past the end of K go through descriptors of
// zero length, which the hardware answers with zeros without touching memory (the stages they land in are never read).
template <class T>
__device__ __forceinline__ void ring_load_one(const RingLoads& L, unsigned char* smem, int slab, int n) {
    const int wrow = L.wrow;
    unsigned char* base = smem + (slab & 1) * T::STAGE_BYTES;
    const int soff = T::PIECES ? piece_offset(L, slab, n < T::RA ? kPieceA : kPieceB) : slab * kRowBytes;
    const bool live = slab < L.KT;
    if (n < T::RA ? T::TRA : T::TRB) {
        // the slab's rows of k: a buffer that begins at them and ends where the operand ends (rows behind it are zeros)
        const bool a = n < T::RA;
        const uint32_t at = (uint32_t)slab * (a ? L.a_slab : L.b_slab), extent = a ? L.a_extent : L.b_extent;
        char* first = (char*)const_cast<void*>(a ? L.base_a : L.base_b0) + at;
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)first, 0, live && at < extent ? (int)(extent - at) : 0, 0x00020000);
        const unsigned voff = a ? L.voff_a[n & 7] : L.voff_b[(n - T::RA) & 7];
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(base + (a ? 0 : T::BM * kRowBytes) + (wrow + (a ? n : n - T::RA) * T::ROWS_PER_PASS) * kRowBytes),
                                                 16, voff, 0, 0, 0);
    } else if (n < T::RA) {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(L.base_a), 0, live ? (int)L.a_extent : 0, 0x00020000);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(base + (wrow + n * T::ROWS_PER_PASS) * kRowBytes), 16,
                                                 L.voff_a[n], soff, 0, 0);
    } else {
        const int m = n - T::RA;
        const bool up_rows = (m * T::ROWS_PER_PASS) % T::WB >= T::WB / 2;
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(up_rows ? L.base_b0 : L.base_b1), 0,
                                                                             live ? (int)L.b_extent : 0, 0x00020000);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(base + T::BM * kRowBytes + (wrow + m * T::ROWS_PER_PASS) * kRowBytes),
                                                 16, L.voff_b[m], soff, 0, 0);
    }
}

// The loads of a task's first two slabs: the weight rows of slab 0 and of slab 1, then the token rows of slab 0 and of
// slab 1 -- weights first because their addresses need no gathered row numbers, so the queue kernel can send them
// off while those are still on their way.  Slab 0 is complete when at most the last RA of them are outstanding.
// Nobody may still be reading the stages (the caller sees to that).
template <class T>
__device__ __forceinline__ void ring_first_weight_loads(const RingLoads& L, unsigned char* smem) {
#pragma unroll
    for (int n = T::RA; n < T::RA + T::RB; ++n) ring_load_one<T>(L, smem, 0, n);
#pragma unroll
    for (int n = T::RA; n < T::RA + T::RB; ++n) ring_load_one<T>(L, smem, 1, n);
}
template <class T>
__device__ __forceinline__ void ring_first_token_load(const RingLoads& L, unsigned char* smem, int q) {   // q = 0..2 RA - 1
    if (q < 2 * T::RA) ring_load_one<T>(L, smem, q / T::RA, q % T::RA);
}
template <class T>
__device__ __forceinline__ void ring_first_loads(const RingLoads& L, unsigned char* smem) {
    ring_first_weight_loads<T>(L, smem);
#pragma unroll
    for (int q = 0; q < 16; ++q) ring_first_token_load<T>(L, smem, q);
}

// The slab loop of a full 256 x 256 tile on four wavefronts of 128 x 128, with the instruction order fixed by hand.
//
// Why not the compiler's order: with one wavefront per SIMD nothing else hides a stall, and the global->LDS loads of
// a slab (64 KB per compute unit) need more than one slab of flight time to stream in at the rate the L2 delivers.
// So (a) both k halves of a slab's fragments are double buffered in registers, which frees the slab's LDS stage at
// mid-slab, (b) the loads of slab kt+2 are issued into that stage right away, two per MFMA row, and stay in flight
// across the barriers (bare s_barrier: a __syncthreads() would wait for them), (c) MFMAs, LDS reads and their
// s_waitcnt are inline asm in the order written by gen_slab_schedule.py (ffn_bf16_slab_steady.inc); the compiler places
// nothing between them but the scalar address updates of the loads.  The accumulators are tied asm operands in
// AGPRs, so they stay put for the whole loop.  Loads use buffer addressing: a 32-bit byte offset per row, computed
// once per task, plus a scalar k offset -- no vector ALU instruction is left in the loop.
// Takes partial row blocks too (the whole tile is computed, rows past the end are not stored).
// Needs: K a multiple of 64 (an odd number of slabs runs one slab of zeros: the loads of slab KT go through descriptors of
// zero length), N a multiple of 64 (columns behind the last one are loaded as zeros and not stored), operand extents
// below 4 GiB.
// On entry the loads of slabs 0 and 1 (ring_first_loads, in that order) are the 32 youngest vector loads of this
// wavefront (stores issued behind them only make the first wait more conservative).  Returns false for a wavefront whose 128 rows are all
// padding: it has taken part in the loads and barriers only and holds no results.
template <class T>
__device__ __forceinline__ bool ring_slabs(int rows, const RingLoads& L, unsigned char* smem, f32x4 (&acc)[8][T::TN]) {
    constexpr int BM = T::BM, STAGE = T::STAGE_BYTES, TN = T::TN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / T::WN, wn = wave % T::WN;
    // The scalar members are the same in every lane; say so here, behind whatever control flow handed L over, or the
    // compiler builds every buffer descriptor in a loop over the lanes.
    RingLoads U = L;
    {
        auto uni = [](unsigned v) { return (unsigned)__builtin_amdgcn_readfirstlane((int)v); };
        auto unip = [&](const void* q) {
            const uint64_t v = (uint64_t)q;
            return (const void*)(((uint64_t)uni((unsigned)(v >> 32)) << 32) | (uint64_t)uni((unsigned)v));
        };
        U.base_a = unip(L.base_a); U.base_b0 = unip(L.base_b0); U.base_b1 = unip(L.base_b1);
        U.a_extent = uni(L.a_extent); U.b_extent = uni(L.b_extent);
        U.a_slab = uni(L.a_slab); U.b_slab = uni(L.b_slab);
        U.piece_slabs = uni(L.piece_slabs); U.piece_recip = uni(L.piece_recip);
        U.KT = (int)uni((unsigned)L.KT); U.wrow = (int)uni((unsigned)L.wrow);
    }
    const int KT = U.KT;                        // an odd one runs one slab more, on the zeros that its loads fetch
    auto load_one = [&](int slab, int n) { ring_load_one<T>(U, smem, slab, n); };

#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    const int frow = lane & 15, fk = lane >> 4;
    const int sw = (frow >> 1) & 7;
    // LDS addresses of this lane's fragment rows: [stage][k half]
    // (the asm reads take raw LDS byte addresses: start from where the dynamic array really begins -- a kernel with
    // static __shared__ variables places it behind them)
    const unsigned lds0 = (unsigned)(__UINTPTR_TYPE__)(lds_void*)smem;
    const unsigned a_row = lds0 + (unsigned)((wm * 128 + frow) * kRowBytes), b_row = lds0 + (unsigned)(BM * kRowBytes + (wn * T::WB + frow) * kRowBytes);
    const unsigned c0 = (unsigned)((fk ^ sw) << 4), c1 = (unsigned)(((4 + fk) ^ sw) << 4);
    const unsigned la0[2] = {a_row + c0, a_row + c1}, lb0[2] = {b_row + c0, b_row + c1};
    const unsigned la1[2] = {la0[0] + STAGE, la0[1] + STAGE}, lb1[2] = {lb0[0] + STAGE, lb0[1] + STAGE};
    // ... and of its turned fragments: [stage][fragment], both k halves within the offset field's reach
    unsigned lat[2][8], lbt[2][TN];
    if constexpr (T::TRA) {
#pragma unroll
        for (int i = 0; i < 8; ++i) lat[1][i] = (lat[0][i] = lds0 + turned_fragment<BM>(wm * 8 + i, lane)) + STAGE;
    }
    if constexpr (T::TRB) {
#pragma unroll
        for (int j = 0; j < TN; ++j) lbt[1][j] = (lbt[0][j] = lds0 + BM * kRowBytes + turned_fragment<T::BN>(wn * TN + j, lane)) + STAGE;
    }
    bf16x8 af[2][8], bfr[2][TN];
    int kt = 0;

#define TURNED(frag, at, pitch, half)                                                                                     \
    do {                                                                                                                 \
        u32x2 lo_, hi_;                                                                                                  \
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(lo_) : "v"(at), "n"((half) * 32 * (pitch)));           \
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(hi_) : "v"(at), "n"((half) * 32 * (pitch) + 4 * (pitch))); \
        frag = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo_, hi_, 0, 1, 2, 3));                                \
    } while (0)
#define MF(i, j, s)                                                                                                      \
    do {                                                                                                                 \
        if constexpr (T::F16) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(bfr[s][j]), "v"(af[s][i])); \
        else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(bfr[s][j]), "v"(af[s][i]));                  \
    } while (0)
#define RA(stg, half, idx)                                                                                               \
    do {                                                                                                                 \
        if constexpr (T::TRA) TURNED(af[half][idx], lat[stg][idx], BM * 2, half);                                        \
        else asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(af[half][idx]) : "v"((stg) ? la1[half] : la0[half]), "n"((idx) * 16 * kRowBytes)); \
    } while (0)
#define RB(stg, half, j)                                                                                                 \
    do {                                                                                                                 \
        if constexpr (T::TRB) TURNED(bfr[half][j], lbt[stg][j], T::BN * 2, half);                                        \
        else asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(bfr[half][j]) : "v"((stg) ? lb1[half] : lb0[half]), "n"((j) * 16 * kRowBytes)); \
    } while (0)
#define WL(n) asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(n))
#define BAR1 do { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); __builtin_amdgcn_s_barrier(); } while (0)
#define BAR2(n) do { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(n) : "memory"); __builtin_amdgcn_s_barrier(); } while (0)
#define GL(n) load_one(kt + 2, n)
#define TAIL asm volatile("s_nop 15\n\ts_nop 3" ::: "memory")
    // Padding rows.  The MFMA pipes run against the board's power limit, so an MFMA on padding rows costs everybody
    // clock.  A wavefront whose 128 rows are all padding (a row block of at most 128 rows: the upper two wavefronts)
    // therefore takes part in the loads and the barriers only: the same slab body with the MFMAs, the fragment reads
    // and their waits left out.  The tile takes as long as before; the layer gains 1 % (Mixtral shape) to 4 % (many
    // small experts) from the clock.  (Skipping the empty 16-row groups of partly filled wavefronts as well, with a
    // scalar branch around their MFMAs, cost more in the full tiles than it returned.)
    if (__builtin_amdgcn_readfirstlane(wm) * 128 >= rows) {
#pragma push_macro("MF")
#pragma push_macro("RA")
#pragma push_macro("RB")
#pragma push_macro("WL")
#undef MF
#undef RA
#undef RB
#undef WL
#define MF(i, j, s) ((void)0)
#define RA(stg, half, idx) ((void)0)
#define RB(stg, half, j) ((void)0)
#define WL(n) ((void)0)
        if constexpr (T::RA == 8) BAR2(8); else BAR2(4);
        for (; kt < KT; kt += 2) {
            {
                constexpr unsigned st = 0, sn = 1;
                (void)st; (void)sn;
#include "ffn_bf16_slab.inc"
            }
            ++kt;
            {
                constexpr unsigned st = 1, sn = 0;
                (void)st; (void)sn;
#include "ffn_bf16_slab.inc"
            }
            --kt;
        }
#pragma pop_macro("WL")
#pragma pop_macro("RB")
#pragma pop_macro("RA")
#pragma pop_macro("MF")
        return false;                           // nothing to store either
    }
    // slab 0 has landed (loads return in issue order; see ring_first_loads)
    if constexpr (T::RA == 8) BAR2(8); else BAR2(4);
    {   // same order as the reads behind BAR2 of a steady-state slab
        constexpr unsigned sn = 0;
        RA(sn, 0, 0);
        RB(sn, 0, 0); RB(sn, 0, 1); RB(sn, 0, 2); RB(sn, 0, 3);
        if constexpr (TN == 8) { RB(sn, 0, 4); RB(sn, 0, 5); RB(sn, 0, 6); RB(sn, 0, 7); }
        RA(sn, 0, 1); RA(sn, 0, 2); RA(sn, 0, 3); RA(sn, 0, 4); RA(sn, 0, 5); RA(sn, 0, 6); RA(sn, 0, 7);
    }
    // Every slab runs the same body, the last two included: their loads (of slabs KT and KT+1) fetch nothing and
    // land in stages nobody reads any more.  Separate tail bodies would be shorter, but between them the compiler is
    // free to spill or copy an accumulator right behind the asm MFMA that writes it, and it does not know that the
    // value is still in flight.
    for (; kt < KT; kt += 2) {
        {
            constexpr unsigned st = 0, sn = 1;
#include "ffn_bf16_slab.inc"
        }
        ++kt;
        {
            constexpr unsigned st = 1, sn = 0;
#include "ffn_bf16_slab.inc"
        }
        --kt;
    }
    // (the TAIL of the last slab also covers the first read of an accumulator behind the loop)
    // The last slab body has read fragments of a slab past the end.  Nobody uses them, so for the compiler their
    // registers are free from here on -- but the reads are still in flight.  Wait for them, and keep the registers
    // occupied until behind that wait.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int i = 0; i < 8; ++i) asm volatile("" ::"v"(af[h][i]));
#pragma unroll
        for (int j = 0; j < TN; ++j) asm volatile("" ::"v"(bfr[h][j]));
    }
#undef MF
#undef RA
#undef RB
#undef WL
#undef BAR1
#undef BAR2
#undef GL
#undef TAIL
#undef TURNED
    return true;
}

// A tile computed as kparts partial sums over the contraction dimension, one task each (the down-projection tiles at the
// end of the task queue: the tasks every workgroup ends its launch with, made short).  Every part stores its fp32
// accumulators (written through: the parts run on any compute unit of the chip), then adds one to the tile's counter;
// the part that finds all the others there runs the epilogue, which adds the parts up in an order that does not depend
// on which part that is (epilogue_full_n_impl), so the result depends on kparts only, never on the schedule.  Returns
// true in that workgroup; every wavefront of the workgroup calls it, `active` false for one whose rows are all padding (it
// keeps the barriers company).
// The buffer has the accumulator layout: [part][wavefront][register group i * TN + j][lane], 16 bytes each; tile_lane is
// this lane's place in part 0.
template <class T>
__device__ __forceinline__ bool partial_tile_arrive(const TaskPtrs& p, unsigned char* smem, f32x4 (&acc)[8][T::TN], bool active,
                                                    float* tile_lane) {
    constexpr int TN = T::TN;
    constexpr size_t kPartFloats = (size_t)T::BM * T::BN;
    static_assert((size_t)T::THREADS / 64 * 8 * TN * 64 * 4 == kPartFloats, "the accumulators of the workgroup are the tile");
    if (active) {
        float* mine = tile_lane + (size_t)p.kpart * kPartFloats;
        const float fill = __int_as_float(0x7FC00000);
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                // (a part whose rows never became ready stores NaN: that is what the tile then holds)
                const f32x4 v = p.poison ? f32x4{fill, fill, fill, fill} : acc[i][j];
                asm volatile(MOE_STORE16_AGENT ::"v"(mine + (i * TN + j) * 256), "v"(v) : "memory");
            }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // this wavefront's part has reached memory
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    int* s_before = reinterpret_cast<int*>(smem + T::NS * T::STAGE_BYTES);    // the staging area is idle until the epilogue
    __syncthreads();
    if (threadIdx.x == 0) *s_before = __hip_atomic_fetch_add(p.part_cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const int before = __builtin_amdgcn_readfirstlane(*s_before);
    __syncthreads();                                      // the word may be overwritten from here on
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    return before == p.kparts - 1;
}

// A task that is a part of a tile, behind its slab loop.
template <class T>
__device__ __forceinline__ void partial_tile_finish(const TaskPtrs& p, unsigned char* smem, f32x4 (&acc)[8][T::TN], bool active) {
    constexpr size_t kPartFloats = (size_t)T::BM * T::BN;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, wave = tid >> 6;
    float* tile_lane = p.part + ((size_t)wave * 8 * T::TN * 64 + lane) * 4;
    if (!partial_tile_arrive<T>(p, smem, acc, active, tile_lane) || !active) return;
    if (p.kparts == 2) {
        const SummedTile<2> parts{tile_lane + (size_t)(1 - p.kpart) * kPartFloats};
        epilogue_full_n_impl<T, 0>(p, smem, acc, NoHook(), parts);
    } else {
        const SummedTile<4> parts{tile_lane};
        epilogue_full_n_impl<T, 0>(p, smem, acc, NoHook(), parts);
    }
}

// One task from start to end: the form the two-launch and the plain-GEMM kernels use.
template <class T>
__device__ __forceinline__ void gemm_tile_ring(const TaskPtrs& p, unsigned char* smem) {
    const RingLoads L = ring_prepare<T>(p);
    __syncthreads();                            // the previous task may still be reading the stages
    ring_first_loads<T>(L, smem);
    f32x4 acc[8][T::TN];
    if (ring_slabs<T>(p.rows, L, smem, acc)) epilogue_full_n<T>(p, smem, acc);
}
// The same for a task that is a part of a tile (TaskPtrs::part).  A copy of its own, slab loop included: with both ends
// behind one loop the compiler reads all accumulators in front of the branch between them and spills what does not fit,
// which costs the whole tiles -- nearly all of them -- 4 to 13 % of their time.
template <class T>
__device__ __forceinline__ void gemm_tile_ring_part(const TaskPtrs& p, unsigned char* smem) {
    const RingLoads L = ring_prepare<T>(p);
    __syncthreads();
    ring_first_loads<T>(L, smem);
    f32x4 acc[8][T::TN];
    const bool active = ring_slabs<T>(p.rows, L, smem, acc);
    partial_tile_finish<T>(p, smem, acc, active);
}

template <class T, bool PARTIAL>
__device__ __forceinline__ void gemm_tile_generic(const TaskPtrs& p, unsigned char* smem) {
    f32x4 acc[T::TM][T::TN];
    mainloop_generic<T, PARTIAL>(p, smem, acc);
    epilogue<T>(p, acc);
}

// The 256 x 256 tile only exists with the hand-ordered slab loop; the host selects it when every task of the launch
// meets that loop's conditions (large_tile_ok) and falls back to the 128 x 128 tile otherwise.
template <class T>
__device__ __forceinline__ void gemm_tile(const TaskPtrs& p, unsigned char* smem) {
    if constexpr (T::HAND) {
        gemm_tile_ring<T>(p, smem);
    } else {
        if (p.rows >= T::BM) gemm_tile_generic<T, false>(p, smem);
        else gemm_tile_generic<T, true>(p, smem);
    }
}

using Tile256 = Tile<256, 256, 2, 2, 2>;
using Tile128x256 = Tile<128, 256, 1, 4, 2>;     // hand-ordered, four wavefronts of 128 x 64 side by side
using Tile256H = Tile<256, 256, 2, 2, 2, true>;  // fp16
using Tile128x256H = Tile<128, 256, 1, 4, 2, true>;
using Tile128 = Tile<128, 128, 2, 2, 2>;         // general loop
using Tile128H = Tile<128, 128, 2, 2, 2, true>;

template <class K>
hipError_t allow_lds(K kernel, int bytes) {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                               bytes);
}

// Which hand-ordered tile a grouped product runs on: the 256 x 256 one or the 128 x 256 one.
//
// The larger tile reads its operands half as often; the smaller one pads less behind an expert's last row and spreads few
// rows over more compute units.  The estimate behind the choice, per projection: row blocks an expert is expected to have
// (rows / height and a half, one if the expert's rows hardly ever reach the height) x column tiles, in rounds over the
// compute units (at least one, and half a round of tail), x the time of a task (tile_task_us).
// Measured, whole layer, 256 x 256 / 128 x 256 / the 128 x 128 tile of the general loop (better of queue and launches):
//   12 experts of 1344 x 2752, GELU: 150 rows each 127 / 112 / 115 us, 444 176 / 168 / 199, 1000 269 / 293 / 350
//   12 experts of 704 x 1152, SwiGLU, 296 rows 107 / 81 / 87;  5 of 1856 x 2112, 200 rows 108 / 78 / 87
//   64 experts of 2048 x 1408, SwiGLU: 93 rows 301 / 279 / 303, 281 492 / 552 / 611
//   8 experts of 4096 x 14336, SwiGLU: 128 rows 775 / 728 / 804, 250 843 / 944 / 1118, 375 1035 / 1252 / 1424
//   16 experts of 2048 x 2048, GELU: 125 rows 133 / 115 / 129, 250 158 / 175 / 195
// The general loop is the fastest of the three at none of them.  The estimate decides all of these pairs as measured but the
// second (444 rows of 1344 x 2752: it takes 256 x 256, 5 % behind), where 264 tasks on 256 compute units are 1.03 rounds, not 1.5.
static double projection_cost(bool large, int64_t pairs, int experts, int column_tiles, int K) {
    const double rows = (double)pairs / experts, height = large ? 256 : 128;
    const double blocks = experts * (rows <= 0.75 * height ? 1.0 : rows / height + 0.5);
    const double rounds = blocks * column_tiles / 256;
    return (rounds <= 1.0 ? 1.0 : rounds + 0.5) * tile_task_us(large, K);
}

}  // namespace
}  // namespace moe355
