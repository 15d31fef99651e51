// Expert FFN in fp32 on the bf16 matrix instructions: every fp32 value as three bf16 pieces that add up to it exactly, the product of
// two values as the six largest of the nine products of their pieces, each exact in fp32 (G. Henry, P. T. P. Tang, A. Heinecke, "Leveraging
// the bfloat16 Artificial Intelligence Datatype for Higher-Precision Computations", ARITH 2019).
//
// v_mfma_f32_32x32x2_f32 multiplies at 157 TFLOP/s, v_mfma_f32_16x16x32_bf16 at 2.5 PFLOP/s: six of the latter for one of the former
// is 2.6 times the rate.  An operand's row holds its pieces one behind the other, [first | second | third] of K each, and a product
// is one contraction of 6 K over pairs of pieces on the hand-ordered tiles of the 16-bit layers (piece_offset, ffn_bf16_tile.hpp);
// only where a slab's loads begin is different.
//
// Precision.  Pieces are rounded to nearest, so the second is at most 2^-8 of the first, the third 2^-8 of the second, and either has
// either sign: the three left-out products are below 2^-22 of a term at the very most, about 2^-27 of it on average, and cancel.
// The sums run from the smallest pairs to the largest, so that the pieces' products are added up before the first pieces' raise the
// rounding error of an addition, and those are added 32 at a time.  Distance from float64 (2-norm), fp32 tile / pieces: the reference's knob file 1.0e-6 / 3.7e-7; 8 experts of 1024 x 2048, GELU, 512 rows each
// 1.1e-6 / 3.6e-7; 16 of 2048 x 1408, SwiGLU, 2048 rows 1.4e-6 / 5.0e-7; one of 1024 x 2048, ReLU, operands of one sign 7.0e-7 / 2.5e-7, all
// equal 6.5e-6 / 1.6e-8, of magnitudes spread over 2^40 5.0e-7 / 3.3e-7, tokens with one value that is not zero 5.7e-7 / 2.1e-7.
// What bounds it: the energy of the bf16 MFMAs on operands whose bits are all random (1.25 PFLOP/s of them, as in a 16-bit layer), so a
// fp32 product runs at 208 TFLOP/s.  The reference's knob file (8192 rows, one expert of 1024 x 4096, ReLU): up and down projection 577 and
// 556 us on the fp32 instructions; 331 and 329 here, on 256- and on 128-row blocks (128 tiles of 256 rows, half the chip: 494), behind 27 us
// for the pieces of tokens and weights at 6.2 TB/s.
// Values are multiplied by 2^24 before they are taken apart, so that the lowest bit of any fp32 number, denormal ones included, is a
// normal bf16 number, and neither the pieces nor the products that matter of small values (2^-62 times 2^-62, say) fall below the
// range; the sums are multiplied by 2^-48.  Values that three pieces do not hold even so -- infinities and NaN, whose products with a
// zero piece would be NaN, and magnitudes of 2^76 and more -- set QueueState::inexact, in the pass that makes the pieces or where the up
// projection's results become some.  So does a sum of either projection that is not finite: the pieces of two values can overflow where
// the product of the values does not (or with the other sign: NaN).  The fp32 tiles at the end (ffn_f32_tile.hip), which do nothing
// otherwise, then take both projections again.  What such a call costs, us, on pieces / on the fp32 tiles without asking / an infinite token /
// sums of 2^76 in the up projection: the knob file 711 / 1067 / 1098 / 1449; 8 experts of 1024 x 2048, SwiGLU, 2048 rows each 1248 / 1825 /
// 1885 / 2571.
#include <algorithm>

#include "f32_pieces_choice.hpp"
#include "ffn_bf16_tile.hpp"
#include "grouped_task.hpp"

namespace moe355 {

hipError_t launch_ffn_f32_tile_if(const FfnArgs&, int phase, const int32_t* only_if, int max_mtiles, int nnt, hipStream_t);   // ffn_f32_tile.hip

namespace {

template <int BM_, int BN_, int WM_, int WN_>
struct PieceTile : Tile<BM_, BN_, WM_, WN_, 2> {
    static constexpr bool PIECES = true;
};
template <int BIG_>
struct PieceSplit {
    static constexpr int BIG = BIG_, BN = 256, THREADS = 256;
    using TH = PieceTile<128, 256, 1, 4>;
    using TB = typename std::conditional<BIG_ == 256, PieceTile<256, 256, 2, 2>, TH>::type;
    static constexpr int LDS_BYTES = TB::LDS_BYTES;
};

constexpr float kPieceScale = 16777216.0f, kSumScale = 1.0f / kPieceScale / kPieceScale;
// Not held by three pieces of kPieceScale times it.
__device__ __forceinline__ bool inexact_as_pieces(float v) { return (__float_as_uint(v) & 0x7FFFFFFFu) >= 0x65800000u; }
static_assert((0x65800000u >> 23) == 127 + 76, "from 2^76 on");
__device__ __forceinline__ bool finite(float v) { return (__float_as_uint(v) & 0x7F800000u) != 0x7F800000u; }
// kPieceScale times two values as pieces: p[i] their i-th pieces side by side.
__device__ __forceinline__ void pieces2(float v0, float v1, uint32_t (&p)[3]) {
    v0 *= kPieceScale;
    v1 *= kPieceScale;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        p[i] = pack2_bf16(v0, v1);
        v0 -= __uint_as_float(p[i] << 16);
        v1 -= __uint_as_float(p[i] & 0xFFFF0000u);
    }
}

// fp32 rows of K -> rows of three pieces, for up to four matrices in one launch; eight values a thread.
struct PieceJob {
    const float* src;
    uint16_t* dst;
    uint32_t vecs;             // groups of eight values (0: none)
    uint32_t row_vecs;         // of a row
    uint32_t first;            // first workgroup of this matrix
};
struct PieceJobs {
    PieceJob job[4];
};
constexpr int kPieceVecs = 2;  // a thread's, 256 apart
__global__ __launch_bounds__(256) void make_pieces_kernel(PieceJobs jobs, int32_t* inexact) {
    int j = 0;
#pragma unroll
    for (int i = 1; i < 4; ++i)
        if (jobs.job[i].vecs && blockIdx.x >= jobs.job[i].first) j = i;
    const PieceJob t = jobs.job[j];
    const uint32_t v0 = (blockIdx.x - t.first) * (256 * kPieceVecs) + threadIdx.x;
    float4 in[kPieceVecs][2];
#pragma unroll
    for (int n = 0; n < kPieceVecs; ++n) {
        const uint32_t v = v0 + 256 * n;
        if (v >= t.vecs) break;
        in[n][0] = reinterpret_cast<const float4*>(t.src)[(size_t)v * 2];
        in[n][1] = reinterpret_cast<const float4*>(t.src)[(size_t)v * 2 + 1];
    }
    bool bad = false;
#pragma unroll
    for (int n = 0; n < kPieceVecs; ++n) {
        const uint32_t v = v0 + 256 * n;
        if (v >= t.vecs) break;
        const float f[8] = {in[n][0].x, in[n][0].y, in[n][0].z, in[n][0].w, in[n][1].x, in[n][1].y, in[n][1].z, in[n][1].w};
        u32x4 out[3];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            uint32_t p[3];
            pieces2(f[2 * w], f[2 * w + 1], p);
            bad = bad || inexact_as_pieces(f[2 * w]) || inexact_as_pieces(f[2 * w + 1]);
#pragma unroll
            for (int i = 0; i < 3; ++i) out[i][w] = p[i];
        }
        const uint32_t row = v / t.row_vecs, col = v - row * t.row_vecs;
        u32x4* d = reinterpret_cast<u32x4*>(t.dst) + (size_t)row * 3 * t.row_vecs + col;
#pragma unroll
        for (int i = 0; i < 3; ++i) d[(size_t)i * t.row_vecs] = out[i];
    }
    if (bad) inexact[0] = 1;
}

// What happens to a tile's sums: UP: bias, activation, and the results as pieces; else bias, and the results in fp32.  A wavefront
// lays 64 of its rows out in its share of the idle slab stages and takes them up again row by row, eight columns a lane, so that the
// activation's library functions stand in the code once and a row is stored in one piece.
struct PieceEpilogue {
    const float* bias0;        // of the output columns, or null
    const float* bias1;        // SwiGLU: the gate's
    float* c;                  // first row of the block, fp32 ...
    uint16_t* c_pieces;        // ... or pieces (UP)
    int N, rows, n0, act;
    int32_t* inexact;
};
template <class T, int EPI, bool UP>
__device__ __forceinline__ void piece_epilogue(const PieceEpilogue& e, unsigned char* smem, f32x4 (&acc)[8][T::TN]) {
    constexpr bool SWIGLU = EPI == MOE_ACT_SWIGLU;
    constexpr int NJ = SWIGLU ? T::TN / 2 : T::TN, COLS = NJ * 16;       // output columns of a wavefront
    constexpr int PITCH = T::TN * 64 + 16;                               // bytes of a laid-out row; 16 neighbouring rows start on different banks
    constexpr int LANES = COLS / 8, ROWS = 64 / LANES;                   // lanes a row, rows a step
    static_assert(4 * 64 * PITCH <= T::LDS_BYTES, "64 rows of every wavefront fit");
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / T::WN, wn = wave % T::WN;
    unsigned char* base = smem + wave * (64 * PITCH);
    unsigned char* put = base + (lane & 15) * PITCH + (lane >> 4) * 16;
    const int sub = lane / LANES, cl = lane % LANES * 8, col = e.n0 + wn * COLS + cl;
    const unsigned char* get = base + sub * PITCH + cl * 4;
    const bool mine = col < e.N;                                         // N is a multiple of 64: eight columns exist together or not at all
    float b0[8], b1[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        b0[i] = e.bias0 && mine ? e.bias0[col + i] : -0.0f;
        b1[i] = SWIGLU && e.bias1 && mine ? e.bias1[col + i] : -0.0f;
    }
    bool bad = false;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < T::TN; ++j) *reinterpret_cast<f32x4*>(put + i * 16 * PITCH + j * 64) = acc[half * 4 + i][j];
        const int row0 = wm * 128 + half * 64 + sub;
#pragma unroll 1
        for (int s = 0; s < 64 / ROWS; ++s) {
            const int row = row0 + s * ROWS;
            bool over = false;
            const f32x4* g = reinterpret_cast<const f32x4*>(get + s * ROWS * PITCH);
            const f32x4* u = SWIGLU ? g + COLS / 4 : g;
            float v[8];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const f32x4 uu = u[q], gg = g[q];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float x = uu[r] * kSumScale + b0[4 * q + r];
                    over = over || !finite(x);           // (here: ReLU makes a zero of -inf.  An infinite gate makes a NaN or stays infinite)
                    if constexpr (SWIGLU) v[4 * q + r] = silu(gg[r] * kSumScale + b1[4 * q + r]) * x;
                    else v[4 * q + r] = act_apply(x, EPI == MOE_ACT_GELU ? MOE_ACT_GELU : e.act);
                }
            }
            if (row >= e.rows || !mine) continue;
            bad = bad || over;
            if constexpr (UP) {
                u32x4 out[3];
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    uint32_t p[3];
                    pieces2(v[2 * w], v[2 * w + 1], p);
                    bad = bad || inexact_as_pieces(v[2 * w]) || inexact_as_pieces(v[2 * w + 1]);
#pragma unroll
                    for (int i = 0; i < 3; ++i) out[i][w] = p[i];
                }
                uint16_t* d = e.c_pieces + (int64_t)row * 3 * e.N + col;
#pragma unroll
                for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x4*>(d + (int64_t)i * e.N) = out[i];
            } else {
                f32x4* d = reinterpret_cast<f32x4*>(e.c + (int64_t)row * e.N + col);
                d[0] = f32x4{v[0], v[1], v[2], v[3]};
                d[1] = f32x4{v[4], v[5], v[6], v[7]};
            }
        }
    }
    if (bad) e.inexact[UP ? 1 : 2] = 1;
}

struct PieceArgs {
    const uint16_t* a_rows;    // pieces of the tokens (with gather) or of the packed rows
    const uint16_t* w;         // pieces of [E, N, K]
    const uint16_t* w1;        // SwiGLU: of the gate's
    const float* bias;
    const float* bias1;
    float* out;
    uint16_t* out_pieces;
    const int32_t* gather;
    const int32_t* count;
    const int32_t* offset;
    int32_t* inexact;
    int E, N, K, act;
    uint32_t a_bytes;
};
// EPI: MOE_ACT_SWIGLU, MOE_ACT_GELU, or MOE_ACT_NONE for PieceArgs::act (none or ReLU).
template <class P, int EPI, bool UP>
__global__ __launch_bounds__(P::THREADS) void ffn_tiled_f32_pieces_kernel(PieceArgs a) {
    constexpr bool SWIGLU = EPI == MOE_ACT_SWIGLU;
    constexpr int COLS = SWIGLU ? P::BN / 2 : P::BN;
    extern __shared__ __align__(16) unsigned char smem[];
    if (a.inexact[0] || (!UP && a.inexact[1])) return;      // (never a word that this launch sets: all wavefronts go the same way)
    GroupedTask t;
    if (!grouped_task<P::BIG>(a.count, a.offset, a.E, (a.N + COLS - 1) / COLS, blockIdx.x, t)) return;
    const int ld = 3 * a.K;
    const int64_t matrix = (int64_t)t.expert * a.N * ld;
    TaskPtrs p{};
    p.a_base = a.a_rows;
    p.gather = a.gather ? a.gather + t.row0 : nullptr;
    p.a_row0 = a.gather ? 0 : t.row0;
    p.a_ld = p.b_ld = ld;
    p.b0 = a.w + matrix;
    p.b1 = SWIGLU ? a.w1 + matrix : nullptr;
    p.N = a.N;
    p.K = 6 * a.K;
    p.rows = t.rows;
    p.n0 = t.ctile * COLS;
    p.swiglu = SWIGLU;
    p.a_extent = a.a_bytes;
    p.b_extent = (uint32_t)((int64_t)a.N * ld * 2);
    const PieceEpilogue e{a.bias ? a.bias + (int64_t)t.expert * a.N : nullptr, SWIGLU && a.bias1 ? a.bias1 + (int64_t)t.expert * a.N : nullptr,
                          UP ? nullptr : a.out + (int64_t)t.row0 * a.N, UP ? a.out_pieces + (int64_t)t.row0 * 3 * a.N : nullptr, a.N, t.rows, p.n0, a.act, a.inexact};
    auto ring = [&](auto tile) {
        using T = decltype(tile);
        const RingLoads L = ring_prepare<T>(p);
        ring_first_loads<T>(L, smem);
        f32x4 acc[8][T::TN];
        const bool mine = ring_slabs<T>(p.rows, L, smem, acc);
        // the stages are the epilogue's from here on: every wavefront has read its fragments, and no load is on its way into them
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        if (mine) piece_epilogue<T, EPI, UP>(e, smem, acc);
    };
    if (P::BIG == 256 && t.rows > 128) ring(typename P::TB());
    else ring(typename P::TH());
}

template <class P, int EPI, bool UP>
hipError_t launch_pieces(const PieceArgs& a, int64_t rows, hipStream_t st) {
    const auto kernel = &ffn_tiled_f32_pieces_kernel<P, EPI, UP>;
    hipError_t e = allow_lds(kernel, P::LDS_BYTES);
    if (e != hipSuccess) return e;
    constexpr int COLS = EPI == MOE_ACT_SWIGLU ? P::BN / 2 : P::BN;
    const int64_t blocks = (rows / P::BIG + a.E) * ((a.N + COLS - 1) / COLS) + kShareSlack;      // no expert has more than rows / BIG + 1 row blocks
    if (blocks > INT32_MAX) return hipErrorInvalidValue;
    kernel<<<(unsigned)blocks, P::THREADS, P::LDS_BYTES, st>>>(a);
    return hipGetLastError();
}
template <int EPI, bool UP>
hipError_t launch_pieces(const PieceArgs& a, int64_t rows, hipStream_t st) {
    const bool large = pieces_large(rows, a.E, (a.N * (EPI == MOE_ACT_SWIGLU ? 2 : 1) + 255) / 256, a.K);
    return large ? launch_pieces<PieceSplit<256>, EPI, UP>(a, rows, st) : launch_pieces<PieceSplit<128>, EPI, UP>(a, rows, st);
}

}  // namespace

// A whole FFN stage.  x_pieces [S, 3, H], w_pieces the matrices [up | down | gate] as pieces, h_pieces [A, 3, I] (may lie on a.h),
// inexact: three words that are zero (QueueState::inexact).
hipError_t launch_ffn_f32_pieces(const FfnArgs& a, const ExpertRows& rows, void* x_pieces, void* w_pieces, void* h_pieces, int32_t* inexact,
                                 int max_mtiles, int nnt0, int nnt1, hipStream_t st) {
    const bool sw = a.act == MOE_ACT_SWIGLU;
    const int64_t A = (int64_t)a.S * a.k, matrices = (int64_t)a.E * a.I * a.H;
    uint16_t* w[3] = {(uint16_t*)w_pieces, (uint16_t*)w_pieces + 3 * matrices, (uint16_t*)w_pieces + 6 * matrices};
    PieceJobs jobs{};
    uint32_t blocks = 0;
    auto add = [&](int i, const void* src, void* dst, int64_t rows_, int K) {
        const int64_t vecs = rows_ * K / 8;
        jobs.job[i] = PieceJob{(const float*)src, (uint16_t*)dst, (uint32_t)vecs, (uint32_t)(K / 8), blocks};
        blocks += (uint32_t)((vecs + 256 * kPieceVecs - 1) / (256 * kPieceVecs));
    };
    add(0, a.x, x_pieces, a.S, a.H);
    add(1, a.w_up, w[0], (int64_t)a.E * a.I, a.H);
    add(2, a.w_down, w[1], (int64_t)a.E * a.H, a.I);
    if (sw) add(3, a.w_gate, w[2], (int64_t)a.E * a.I, a.H);
    make_pieces_kernel<<<blocks, 256, 0, st>>>(jobs, inexact);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    PieceArgs p{(const uint16_t*)x_pieces, w[0], w[2], (const float*)a.b_up, (const float*)a.b_gate, nullptr, (uint16_t*)h_pieces, a.token_indices,
                rows.count, rows.offset, inexact, a.E, a.I, a.H, a.act, (uint32_t)((int64_t)a.S * 3 * a.H * 2)};
    e = sw ? launch_pieces<MOE_ACT_SWIGLU, true>(p, A, st) : a.act == MOE_ACT_GELU ? launch_pieces<MOE_ACT_GELU, true>(p, A, st) : launch_pieces<MOE_ACT_NONE, true>(p, A, st);
    if (e != hipSuccess) return e;
    p = PieceArgs{(const uint16_t*)h_pieces, w[1], nullptr, (const float*)a.b_down, nullptr, (float*)a.y, nullptr, nullptr,
                  rows.count, rows.offset, inexact, a.E, a.H, a.I, MOE_ACT_NONE, (uint32_t)(A * 3 * a.I * 2)};
    e = launch_pieces<MOE_ACT_NONE, false>(p, A, st);
    if (e != hipSuccess) return e;
    e = launch_ffn_f32_tile_if(a, 0, inexact, max_mtiles, nnt0, st);      // (behind the last reader of h_pieces, on which it may write)
    if (e != hipSuccess) return e;
    return launch_ffn_f32_tile_if(a, 1, inexact, max_mtiles, nnt1, st);
}

}  // namespace moe355
