// Router stage: gate logits, top-k selection and gate weights.
//
// The reference has no router (its config macros E_TOP_K / NUM_EXPERTS are defined at
// CMakeLists.txt:207,213 and never read), so the semantics are this library's:
//   logits[t,e] = sum_k x[t,k] * gate_w[e,k] (+ gate_bias[e]) with gate_w [E,H] row-major, the (N,K)
//   operand convention of the reference GEMM (mma.cuh:417-419).
// The fp32 summation order is fixed so that the integer routing results are reproducible bit for bit:
// lane l of a wavefront owns partial sum l and takes, in ascending k, every k with (k/8) % 64 == l using
// one fmaf per element; the 64 partials are folded by an xor butterfly (32,16,8,4,2,1); the bias is added
// last.  Top-k is taken on the logits (softmax and sigmoid are monotone), ties to the lower expert index.
#include <algorithm>
#include <type_traits>
#include <cstdlib>

#include "moe_internal.hpp"
#include "topk.hpp"

namespace moe355 {
namespace {

__device__ __forceinline__ void load8(const float* p, float (&v)[8]) {
    const float4 a = reinterpret_cast<const float4*>(p)[0];
    const float4 b = reinterpret_cast<const float4*>(p)[1];
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
// two 16-bit values packed in a dword -> fp32 (exact)
__device__ __forceinline__ float lo16(uint32_t w, bf16_s) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float hi16(uint32_t w, bf16_s) { return __uint_as_float(w & 0xFFFF0000u); }
__device__ __forceinline__ float lo16(uint32_t w, f16_s) { return (float)__builtin_bit_cast(_Float16, (uint16_t)(w & 0xFFFFu)); }
__device__ __forceinline__ float hi16(uint32_t w, f16_s) { return (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16)); }

template <typename T16>
__device__ __forceinline__ void load8(const T16* p, float (&v)[8]) {
    const uint4 a = reinterpret_cast<const uint4*>(p)[0];
    v[0] = lo16(a.x, T16{}); v[1] = hi16(a.x, T16{});
    v[2] = lo16(a.y, T16{}); v[3] = hi16(a.y, T16{});
    v[4] = lo16(a.z, T16{}); v[5] = hi16(a.z, T16{});
    v[6] = lo16(a.w, T16{}); v[7] = hi16(a.w, T16{});
}

// Folds the 64 per-lane partial sums of 16 independent sums at once.  At xor distance 32, 16, 8, 4 a lane keeps one
// register of each pair and hands the other to its partner (halving the registers per step), then distances 2 and 1
// on the one register left.  Each sum adds lane l to lane l ^ d for d = 32, 16, 8, 4, 2, 1 in that order: the result
// has the bits of the plain butterfly.  Returns the sum of red[index] with index = fold16_index(lane), valid in the
// lanes with (lane & 3) == 0.
// The exchanges stay in the vector ALU: v_permlane32_swap / v_permlane16_swap trade the halves (the odd 16-lane rows)
// of a register pair, which is the keep-one-hand-over-the-other step in one instruction; distances 8 .. 1 are DPP
// moves (row rotate by 8; row shifts by 4 under bank masks; quad permutes).  Through the LDS crossbar (ds_bpermute)
// the seventeen exchanges of a fold cost about as much as a quarter of the multiply-adds they follow.
template <int CTRL, int BANKS = 0xF>
__device__ __forceinline__ float dpp_from(float old, float v) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(__float_as_uint(old), __float_as_uint(v), CTRL, 0xF, BANKS, false));
}
__device__ __forceinline__ float lane_xor8(float v) { return dpp_from<0x128>(0.0f, v); }                    // row_ror:8
__device__ __forceinline__ float lane_xor4(float v) { return dpp_from<0x114, 0xA>(dpp_from<0x104, 0x5>(0.0f, v), v); }   // row_shl:4 | row_shr:4
__device__ __forceinline__ float lane_xor2(float v) { return dpp_from<0x4E>(0.0f, v); }                     // quad_perm [2,3,0,1]
__device__ __forceinline__ float lane_xor1(float v) { return dpp_from<0xB1>(0.0f, v); }                     // quad_perm [1,0,3,2]

__device__ __forceinline__ float fold16(float (&red)[16], int lane) {
    typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int i = 0; i < 8; ++i) {      // distance 32: lanes 0..31 keep red[2i], lanes 32..63 keep red[2i+1]
        const u32x2_t r = __builtin_amdgcn_permlane32_swap(__float_as_uint(red[2 * i]), __float_as_uint(red[2 * i + 1]), false, false);
        red[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {      // distance 16: even 16-lane rows keep red[2i], odd rows red[2i+1]
        const u32x2_t r = __builtin_amdgcn_permlane16_swap(__float_as_uint(red[2 * i]), __float_as_uint(red[2 * i + 1]), false, false);
        red[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    {
        const bool hi = (lane & 8) != 0;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const float keep = hi ? red[2 * i + 1] : red[2 * i];
            const float send = hi ? red[2 * i] : red[2 * i + 1];
            red[i] = keep + lane_xor8(send);
        }
    }
    {
        const bool hi = (lane & 4) != 0;
        const float keep = hi ? red[1] : red[0];
        const float send = hi ? red[0] : red[1];
        red[0] = keep + lane_xor4(send);
    }
    float sum = red[0];
    sum = sum + lane_xor2(sum);
    sum = sum + lane_xor1(sum);
    return sum;
}
__device__ __forceinline__ int fold16_index(int lane) {
    return ((lane >> 5) & 1) | (((lane >> 4) & 1) << 1) | (((lane >> 3) & 1) << 2) | (((lane >> 2) & 1) << 3);
}

// A wavefront keeps TPW token rows in registers (lane l owns the 8-element chunks l, l+64, ... of each row, as
// fp32) and walks over its share of the experts: one 16-byte load of the expert's row per chunk feeds 8*TPW
// fmafs; the 64 partial sums of 16 (token, expert) pairs are folded together (see the loop).  grid = (token groups of 4*TPW, expert chunks); NCH = chunks per lane = ceil(H / 512).
template <typename T, int NCH, int TPW>
__global__ __launch_bounds__(256) void gate_logits_kernel(const T* __restrict__ x, const T* __restrict__ gate_w,
                                                          const float* __restrict__ gate_bias,
                                                          float* __restrict__ logits, int S, int H, int E,
                                                          int experts_per_block) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int t0 = (blockIdx.x * 4 + wave) * TPW;
    if (t0 >= S) return;
    const int nchunk = H >> 3;
    float xr[TPW][NCH][8];
#pragma unroll
    for (int q = 0; q < TPW; ++q) {
        const int t = min(t0 + q, S - 1);          // a ragged last group recomputes the last token; not stored
#pragma unroll
        for (int j = 0; j < NCH; ++j) {
            const int c = lane + j * kWave;
            if (c < nchunk) load8(x + (size_t)t * H + c * 8, xr[q][j]);
            else {
#pragma unroll
                for (int v = 0; v < 8; ++v) xr[q][j][v] = 0.0f;
            }
        }
    }
    const int e0 = blockIdx.y * experts_per_block;
    const int e1 = min(E, e0 + experts_per_block);
    // raw 16-byte chunks of the next expert's row are fetched while the current expert is being summed
    typedef unsigned int raw_t __attribute__((ext_vector_type(sizeof(T) == 4 ? 8 : 4)));
    raw_t wn[NCH];
    auto fetch = [&](int e) {
        const T* wr = gate_w + (size_t)e * H;
#pragma unroll
        for (int j = 0; j < NCH; ++j) {
            const int c = lane + j * kWave;
            if (c < nchunk) wn[j] = *reinterpret_cast<const raw_t*>(wr + c * 8);
        }
    };
    fetch(e0);
    // Experts are taken EG at a time so that EG * TPW = 16 partial-sum registers are folded together: at xor
    // distance 32, 16, 8, 4 a lane keeps one register of each pair and hands the other to its partner, which
    // halves the registers per step instead of running six shuffles per sum.  Every sum still adds lane l to
    // lane l ^ d for d = 32, 16, 8, 4, 2, 1 in that order, so the result is bit-identical to the plain butterfly.
    constexpr int EG = 16 / TPW;
    for (int eb = e0; eb < e1; eb += EG) {
        float red[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) red[r] = 0.0f;
#pragma unroll
        for (int g = 0; g < EG; ++g) {
            const int e = eb + g;
            if (e >= e1) break;
            raw_t wc[NCH];
#pragma unroll
            for (int j = 0; j < NCH; ++j) wc[j] = wn[j];
            if (e + 1 < e1) fetch(e + 1);
#pragma unroll
            for (int j = 0; j < NCH; ++j) {
                const int c = lane + j * kWave;
                if (c < nchunk) {
                    float wv[8];
                    if constexpr (sizeof(T) == 4) {
#pragma unroll
                        for (int v = 0; v < 8; ++v) wv[v] = __uint_as_float(wc[j][v]);
                    } else {
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            wv[2 * v] = lo16(wc[j][v], T{});
                            wv[2 * v + 1] = hi16(wc[j][v], T{});
                        }
                    }
#pragma unroll
                    for (int q = 0; q < TPW; ++q)
#pragma unroll
                        for (int v = 0; v < 8; ++v)
                            red[g * TPW + q] = __builtin_fmaf(xr[q][j][v], wv[v], red[g * TPW + q]);
                }
            }
        }
        const float sum = fold16(red, lane);
        const int r = fold16_index(lane);
        const int e = eb + r / TPW, t = t0 + r % TPW;
        if ((lane & 3) == 0 && e < e1 && t < S) logits[(size_t)t * E + e] = gate_bias ? sum + gate_bias[e] : sum;
    }
}

template <typename T, int NCH, int TPW>
hipError_t launch_gate_variant(const void* x, const void* gate_w, const float* gate_bias, float* logits, int S, int H,
                               int E, hipStream_t st) {
    const int token_blocks = (S + 4 * TPW - 1) / (4 * TPW);
    // enough workgroups to occupy the chip even when S is small (decode shapes)
    int chunks = 1;
    while (token_blocks * chunks < 1024 && chunks < E) chunks *= 2;
    const int per = (E + chunks - 1) / chunks;
    chunks = (E + per - 1) / per;
    gate_logits_kernel<T, NCH, TPW><<<dim3(token_blocks, chunks), 256, 0, st>>>((const T*)x, (const T*)gate_w,
                                                                                gate_bias, logits, S, H, E, per);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_gate_typed(const void* x, const void* gate_w, const float* gate_bias, float* logits, int S, int H,
                             int E, hipStream_t st) {
    const bool many = (int64_t)S * E >= 4 * 4096;   // enough (token, expert) work to give each wavefront 4 tokens
    if (H <= 1024) return many ? launch_gate_variant<T, 2, 4>(x, gate_w, gate_bias, logits, S, H, E, st)
                               : launch_gate_variant<T, 2, 1>(x, gate_w, gate_bias, logits, S, H, E, st);
    if (H <= 2048) return many ? launch_gate_variant<T, 4, 4>(x, gate_w, gate_bias, logits, S, H, E, st)
                               : launch_gate_variant<T, 4, 1>(x, gate_w, gate_bias, logits, S, H, E, st);
    if (H <= 4096) return many ? launch_gate_variant<T, 8, 2>(x, gate_w, gate_bias, logits, S, H, E, st)
                               : launch_gate_variant<T, 8, 1>(x, gate_w, gate_bias, logits, S, H, E, st);
    if (H <= 8192) return launch_gate_variant<T, 16, 1>(x, gate_w, gate_bias, logits, S, H, E, st);
    if (H <= 16384) return launch_gate_variant<T, 32, 1>(x, gate_w, gate_bias, logits, S, H, E, st);
    return hipErrorInvalidValue;
}

// ---- second logits kernel: register tiles of (tokens x experts), K streamed ----
//
// The kernel above keeps whole token rows in registers and walks the experts one after the other, one 16-byte load
// in flight per chunk: with many experts or few tokens it waits on memory latency most of the time.  Here a wavefront
// owns TT tokens x TE experts (TT * TE running sums per lane), walks K in steps of one 8-element chunk per lane
// (chunk c = lane + 64 j, exactly the elements partial sum `lane` takes), and has the TT + TE loads of the next step
// in flight while it works on the current one.  Every sum sees the same fmaf sequence and the same fold as above, so
// the logits are bit-identical.  A workgroup is WT x WE wavefronts over (tokens, experts); neighbouring wavefronts
// read the same rows at the same time and share them in the compute unit's L1.
template <typename T>
struct RawChunk {
    typedef unsigned int type __attribute__((ext_vector_type(sizeof(T) == 4 ? 8 : 4)));
};

template <typename T>
__device__ __forceinline__ void widen8(const typename RawChunk<T>::type& r, float (&v)[8]) {
    if constexpr (sizeof(T) == 4) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = __uint_as_float(r[i]);
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[2 * i] = lo16(r[i], T{});
            v[2 * i + 1] = hi16(r[i], T{});
        }
    }
}

// The token's top-k selection right behind its sums (FUSE): when the workgroup's WE x TE expert columns cover every
// expert, the logits of its WT x TT tokens meet in LDS and each wavefront selects for its share of the tokens with the
// very function the stand-alone top-k kernel runs -- one launch less, and the logits go to memory only when the caller
// asked for them (`logits` may then be null).
struct GateTopk {
    int32_t* idx;       // [S, k]
    float* w;           // [S, k]
    int k, gate_fn, norm;
};

template <typename T, int TT, int TE, int WT, int WE, bool FUSE>
__global__ __launch_bounds__(WT * WE * 64) void gate_tile_kernel(const T* __restrict__ x, const T* __restrict__ gate_w,
                                                                 const float* __restrict__ gate_bias,
                                                                 float* __restrict__ logits, int S, int H, int E,
                                                                 GateTopk tk) {
    static_assert((TT * TE) % 16 == 0 && 16 % TT == 0, "sums are folded sixteen at a time: TT tokens x 16/TT experts");
    typedef typename RawChunk<T>::type raw_t;
    constexpr int ECOLS = WE * TE;                        // expert columns of a workgroup
    __shared__ float s_log[FUSE ? WT * TT * ECOLS : 1];   // [token of the workgroup][expert]
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int t0 = (blockIdx.x * WT + wave / WE) * TT, e0 = (blockIdx.y * WE + wave % WE) * TE;
    const bool live = t0 < S && e0 < E;
    if (!FUSE && !live) return;
    if (live) {
        const int nchunk = H >> 3, nstep = (nchunk + kWave - 1) / kWave;
        const T* xrow[TT];
        const T* wrow[TE];
#pragma unroll
        for (int q = 0; q < TT; ++q) xrow[q] = x + (size_t)min(t0 + q, S - 1) * H + lane * 8;    // rows past the end are
#pragma unroll
        for (int g = 0; g < TE; ++g) wrow[g] = gate_w + (size_t)min(e0 + g, E - 1) * H + lane * 8;   // computed, not stored
        float acc[TT][TE];
#pragma unroll
        for (int q = 0; q < TT; ++q)
#pragma unroll
            for (int g = 0; g < TE; ++g) acc[q][g] = 0.0f;
        raw_t xn[TT], wn[TE];
        auto fetch = [&](int j) {
            if (lane + j * kWave < nchunk) {
#pragma unroll
                for (int q = 0; q < TT; ++q) xn[q] = *reinterpret_cast<const raw_t*>(xrow[q] + (size_t)j * (kWave * 8));
#pragma unroll
                for (int g = 0; g < TE; ++g) wn[g] = *reinterpret_cast<const raw_t*>(wrow[g] + (size_t)j * (kWave * 8));
            }
        };
        fetch(0);
        for (int j = 0; j < nstep; ++j) {
            raw_t xc[TT], wc[TE];
#pragma unroll
            for (int q = 0; q < TT; ++q) xc[q] = xn[q];
#pragma unroll
            for (int g = 0; g < TE; ++g) wc[g] = wn[g];
            if (j + 1 < nstep) fetch(j + 1);
            if (lane + j * kWave < nchunk) {      // partial sum `lane` takes chunk lane + 64 j only if the row has it
                float xv[TT][8];
#pragma unroll
                for (int q = 0; q < TT; ++q) widen8<T>(xc[q], xv[q]);
#pragma unroll
                for (int g = 0; g < TE; ++g) {
                    float wv[8];
                    widen8<T>(wc[g], wv);
#pragma unroll
                    for (int q = 0; q < TT; ++q)
#pragma unroll
                        for (int v = 0; v < 8; ++v) acc[q][g] = __builtin_fmaf(xv[q][v], wv[v], acc[q][g]);
                }
            }
        }
        constexpr int EG = 16 / TT;       // experts per fold
        const int r = fold16_index(lane);
#pragma unroll
        for (int gb = 0; gb < TE; gb += EG) {
            float red[16];
#pragma unroll
            for (int g = 0; g < EG; ++g)
#pragma unroll
                for (int q = 0; q < TT; ++q) red[g * TT + q] = acc[q][gb + g];
            const float sum = fold16(red, lane);
            const int e = e0 + gb + r / TT, t = t0 + r % TT;
            if ((lane & 3) == 0 && e < E && t < S) {
                const float val = gate_bias ? sum + gate_bias[e] : sum;
                if (!FUSE || logits) logits[(size_t)t * E + e] = val;
                if (FUSE) s_log[((wave / WE) * TT + r % TT) * ECOLS + e] = val;     // one expert tile per row: e < ECOLS
            }
        }
    }
    if constexpr (FUSE) {
        __syncthreads();
        for (int q = wave; q < WT * TT; q += WT * WE) {   // this wavefront's share of the workgroup's tokens
            const int t = blockIdx.x * (WT * TT) + q;
            if (t < S) topk_one_token<1>(s_log + q * ECOLS, t, E, tk.k, tk.gate_fn, tk.norm, tk.idx, tk.w, lane);
        }
    }
}

// Returns through *fused whether the launch also selected (tk non-null and every expert in one workgroup's columns).
template <typename T, int TT, int TE, int WT, int WE>
hipError_t launch_gate_tile(const void* x, const void* gate_w, const float* gate_bias, float* logits, bool keep_logits,
                            int S, int H, int E, const GateTopk* tk, bool* fused, hipStream_t st) {
    const dim3 grid((S + WT * TT - 1) / (WT * TT), (E + WE * TE - 1) / (WE * TE));
    if (tk && grid.y == 1) {
        gate_tile_kernel<T, TT, TE, WT, WE, true><<<grid, WT * WE * 64, 0, st>>>((const T*)x, (const T*)gate_w, gate_bias,
                                                                                keep_logits ? logits : nullptr, S, H, E, *tk);
        *fused = true;
    } else {
        gate_tile_kernel<T, TT, TE, WT, WE, false><<<grid, WT * WE * 64, 0, st>>>((const T*)x, (const T*)gate_w, gate_bias,
                                                                                 logits, S, H, E, GateTopk{});
    }
    return hipGetLastError();
}

// Tile choice: big tiles when there are enough (token, expert) pairs to fill the chip with them, small ones when
// the layer is decode-sized and only more wavefronts bring more loads in flight; a 4 x 1 wavefront arrangement when
// the experts fit one wavefront's tile.
template <typename T>
hipError_t launch_gate_tiled(const void* x, const void* gate_w, const float* gate_bias, float* logits, bool keep_logits,
                             int S, int H, int E, int opt_tile, const GateTopk* tk, bool* fused, hipStream_t st) {
    const int64_t pairs = (int64_t)S * E;
    int variant = pairs >= 32768 ? 0 : 1;
    if (opt_tile >= 0 && opt_tile <= 2) variant = opt_tile;
#define MOE355_GATE_TILE_ARGS x, gate_w, gate_bias, logits, keep_logits, S, H, E, tk, fused, st
    switch (variant) {
        case 0:
            return E <= 8 ? launch_gate_tile<T, 4, 8, 4, 1>(MOE355_GATE_TILE_ARGS) : launch_gate_tile<T, 4, 8, 2, 2>(MOE355_GATE_TILE_ARGS);
        case 1:
            return E <= 4 ? launch_gate_tile<T, 4, 4, 4, 1>(MOE355_GATE_TILE_ARGS) : launch_gate_tile<T, 4, 4, 2, 2>(MOE355_GATE_TILE_ARGS);
        default:
            return E <= 8 ? launch_gate_tile<T, 2, 8, 4, 1>(MOE355_GATE_TILE_ARGS) : launch_gate_tile<T, 2, 8, 2, 2>(MOE355_GATE_TILE_ARGS);
    }
#undef MOE355_GATE_TILE_ARGS
}

// ---- third logits kernel: the same sums on the matrix cores (16-bit layers, H a multiple of 512) ----
//
// v_mfma_f32_16x16x1_4b_f32 is four independent 16 x 16 outer products with k = 1: D_b[i][j] = C_b[i][j] + A_b[i] B_b[j],
// one multiply-add per element -- and the product of two bf16 (or fp16) values is exact in fp32, so each element sees
// exactly the fmaf the kernels above perform, at the full fp32 rate of the matrix pipe (twice the unpacked vector rate).
// A tile is 16 tokens x 16 experts.  Block b of accumulator g carries partial sum p = 4 g + b of every pair of the tile: lane
// 16 b + i reads the 16-byte chunk p + 64 j of token row i (and of expert row i) -- the chunk partial sum p takes in step j, i.e.
// elements 32 (16 j + g) + 8 b onwards -- and its 8 elements go through 8 MFMAs in ascending k.  The even g belong to one
// wavefront of a pair and the odd g to the other (8 accumulators = 128 registers each, so two wavefronts fit a SIMD).  The 32
// partial sums a wavefront holds of a pair sit in one lane (accumulator g, register 4 b + r: token 4 (lane / 16) + r, expert
// lane % 16): p is folded with p + 32, 16 and 8 (g with g + 8, 4, 2) in the lane, with p + 4 (g with g + 1) across the two
// wavefronts through LDS, then with p + 2 and p + 1 (b) in the lane again -- the pairings of fold16, so the logits are bit-identical.
//
// A workgroup holds 2 x 2 tiles (32 tokens x 32 experts).  A step's 64 rows of 1 KiB go from memory straight into one of two stages,
// requested two steps ahead and across the end of a tile too: the workgroups stay, `tiles` of them in steps of the grid.  What bounds
// it: a SIMD's two wavefronts share the pipe, and the two widening operations an MFMA needs do not run beside fp32 MFMAs (measured on
// registers: 36 cycles an MFMA without, 48 with them; 64 here).  16384 tokens x 64 experts of 2048 75.6 -> 72.0 us in a trace,
// against rows fetched into registers, 64 bytes of each of 16 a request, one tile's column of 32 experts a workgroup; with the selection
// (topk16_kernel) behind it 81 -> 69 us a call, 8192 tokens 42 -> 36, 4000 30.5 -> 22.2; 1024 tokens x 256 of 7168 74 -> 55.  Few tiles, which AUTO
// leaves to the kernels above, were faster as they were: 1000 tokens x 64 experts 15.4 -> 20.4 with option gate_mfma = 1.
typedef float gate_f32x16 __attribute__((ext_vector_type(16)));

template <typename T>
struct GateStage {
    static constexpr int TT = 2, ET = 2;                     // tiles of a workgroup: tokens, experts
    static constexpr int WAVES = TT * ET * 2, THREADS = WAVES * 64, ROWS = (TT + ET) * 16, PER = ROWS / WAVES;
    static constexpr int STAGE_BYTES = ROWS * 1024, FOLD = 8, FOLD_BYTES = WAVES * FOLD * 64 * 4;
    static constexpr int LDS_BYTES = 2 * STAGE_BYTES + FOLD_BYTES;
    static_assert(LDS_BYTES <= 160 * 1024 && ROWS % WAVES == 0, "two stages and the folds");
};
typedef __attribute__((address_space(3))) void gate_lds_void;
typedef const __attribute__((address_space(1))) void gate_gbl_void;

template <typename T>
__global__ __launch_bounds__(GateStage<T>::THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void gate_mfma_kernel(
    const T* __restrict__ x, const T* __restrict__ gate_w, const float* __restrict__ gate_bias, float* __restrict__ logits, int S, int H, int E,
    int etiles, int tiles) {
    using G = GateStage<T>;
    typedef typename RawChunk<T>::type raw_t;
    constexpr int TT = G::TT, ET = G::ET, NG = 8, ECOLS = ET * 16;
    extern __shared__ __align__(16) unsigned char smem[];
    float* s_fold = reinterpret_cast<float*>(smem + 2 * G::STAGE_BYTES);                       // [wavefront][2 b + r][lane]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = wave % 2, ei = wave / 2 % ET, ti = wave / (2 * ET);      // q: this wavefront's parity of g
    const int b = lane >> 4, i = lane & 15;
    const int nstep = H / 512;
    // Tile id -> token tile and expert tile: the expert tiles of the same tokens are eight ids apart, on one XCD and close in time.
    auto place = [&](int id, int& t0, int& e0) {
        const int group = id >> 3, tt = group / etiles * 8 + (id & 7);
        t0 = tt * TT * 16;
        e0 = group % etiles * ECOLS;
        return t0 < S;
    };
    auto next_tile = [&](int id, int& t0, int& e0) {
        while (id < tiles && !place(id, t0, e0)) id += gridDim.x;
        return id;
    };
    // Row r of a stage: its 16-byte chunk c lies at c ^ (r & 15), so that the sixteen rows of a fragment read meet all banks.
    auto request = [&](int t0, int e0, int step, int stage) {
#pragma unroll
        for (int n = 0; n < G::PER; ++n) {
            const int r = wave + n * G::WAVES;
            const T* row = r < TT * 16 ? x + (size_t)min(t0 + r, S - 1) * H : gate_w + (size_t)min(e0 + r - TT * 16, E - 1) * H;
            __builtin_amdgcn_global_load_lds((gate_gbl_void*)(row + step * 512 + ((lane ^ (r & 15)) << 3)),
                                             (gate_lds_void*)(smem + stage * G::STAGE_BYTES + r * 1024), 16, 0, 0);
        }
    };
    const unsigned lds0 = (unsigned)(__UINTPTR_TYPE__)(gate_lds_void*)smem;
    const unsigned xa = lds0 + (ti * 16 + i) * 1024 + ((b ^ i) << 4), wa = lds0 + ((TT + ei) * 16 + i) * 1024 + ((b ^ i) << 4);

    int t0, e0, id = next_tile(blockIdx.x, t0, e0);
    if (id >= tiles) return;
    // the step that is requested next
    int rt0 = t0, re0 = e0, rid = id, rstep = 0;
    auto advance = [&]() {
        if (++rstep == nstep) {
            rstep = 0;
            rid = next_tile(rid + gridDim.x, rt0, re0);
        }
    };
    int stage = 0, on_the_way = 0;
    for (; on_the_way < 2 && rid < tiles; ++on_the_way) {
        request(rt0, re0, rstep, on_the_way);
        advance();
    }
    while (true) {
        gate_f32x16 acc[NG];
#pragma unroll
        for (int m = 0; m < NG; ++m)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[m][v] = 0.f;
        for (int j = 0; j < nstep; ++j) {
            // (stores of the tile before are younger than both steps' requests: they only make the wait more cautious)
            if (on_the_way < 2) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(G::PER) : "memory");
            __builtin_amdgcn_s_barrier();
            const unsigned at = stage * G::STAGE_BYTES;
#pragma unroll
            for (int m = 0; m < NG; m += 4) {       // four accumulators at a time: consecutive MFMAs are independent
                raw_t xr[4], wr[4];
                unsigned ax[4], aw[4];
#pragma unroll
                for (int h = 0; h < 4; ++h) {
                    const unsigned g = (q + 2 * (m + h)) << 6;
                    ax[h] = (xa ^ g) + at;
                    aw[h] = (wa ^ g) + at;
                }
                asm volatile("ds_read_b128 %0, %8\n\tds_read_b128 %1, %9\n\tds_read_b128 %2, %10\n\tds_read_b128 %3, %11\n\t"
                             "ds_read_b128 %4, %12\n\tds_read_b128 %5, %13\n\tds_read_b128 %6, %14\n\tds_read_b128 %7, %15\n\ts_waitcnt lgkmcnt(0)"
                             : "=&v"(xr[0]), "=&v"(wr[0]), "=&v"(xr[1]), "=&v"(wr[1]), "=&v"(xr[2]), "=&v"(wr[2]), "=&v"(xr[3]), "=&v"(wr[3])
                             : "v"(ax[0]), "v"(aw[0]), "v"(ax[1]), "v"(aw[1]), "v"(ax[2]), "v"(aw[2]), "v"(ax[3]), "v"(aw[3])
                             : "memory");
                float xv[4][8], wv[4][8];
#pragma unroll
                for (int h = 0; h < 4; ++h) {
                    widen8<T>(xr[h], xv[h]);
                    widen8<T>(wr[h], wv[h]);
                }
#pragma unroll
                for (int v = 0; v < 8; ++v)
#pragma unroll
                    for (int h = 0; h < 4; ++h) acc[m + h] = __builtin_amdgcn_mfma_f32_16x16x1f32(xv[h][v], wv[h][v], acc[m + h], 0, 0, 0);
            }
            __builtin_amdgcn_s_barrier();           // the stage is free
            if (rid < tiles) {
                request(rt0, re0, rstep, stage);
                advance();
            } else {
                --on_the_way;
            }
            stage ^= 1;
        }
        // acc[m] holds g = 2 m + q: g + 8, g + 4, g + 2 are m + 4, m + 2, m + 1
        float u[16];
#pragma unroll
        for (int v = 0; v < 16; ++v)      // p with p + 32, then p + 16, then p + 8
            u[v] = ((acc[0][v] + acc[4][v]) + (acc[2][v] + acc[6][v])) + ((acc[1][v] + acc[5][v]) + (acc[3][v] + acc[7][v]));
        // each wavefront of the pair goes on with two of the four tokens r of every lane
        float* mine = s_fold + wave * G::FOLD * 64 + lane;
#pragma unroll
        for (int bb = 0; bb < 4; ++bb)
#pragma unroll
            for (int rr = 0; rr < 2; ++rr) mine[(2 * bb + rr) * 64] = q ? u[4 * bb + rr] : u[4 * bb + 2 + rr];
        __syncthreads();
        const float* other = s_fold + (wave ^ 1) * G::FOLD * 64 + lane;
#pragma unroll
        for (int rr = 0; rr < 2; ++rr) {
            const int r = q * 2 + rr;
            float s[4];
#pragma unroll
            for (int bb = 0; bb < 4; ++bb) s[bb] = (q ? u[4 * bb + 2 + rr] : u[4 * bb + rr]) + other[(2 * bb + rr) * 64];     // ... p + 4
            const float sum = (s[0] + s[2]) + (s[1] + s[3]);                                                       // ... p + 2, p + 1
            const int t = t0 + ti * 16 + 4 * b + r, e = e0 + ei * 16 + i;
            if (t < S && e < E) {
                const float val = gate_bias ? sum + gate_bias[e] : sum;
                logits[(size_t)t * E + e] = val;
            }
        }
        id = next_tile(id + gridDim.x, t0, e0);
        if (id >= tiles) return;
        __syncthreads();                            // the folds have been read
    }
}
// The matrix-core kernel takes 16-bit layers whose rows split into full steps of 512 elements, from 150 workgroups' tiles on that the
// experts fill to three quarters, or where they are many and the experts fill most of 16 columns.  This / the best other kernel, us,
// selection included, rows of 2048: 64 experts, 2500 tokens (158) 21.0 / 22.7, 2000 (126) 20.5 / 19.2; 32 experts, 8192 tokens (256) 20.8 /
// 28.2, 4096 (128) 18.4 / 16.5; 24 experts, 16384 (512) 36.3 / 46.7; 128, 4096 (512) 34.8 / 49.3; 256 experts of 7168, 1024 tokens (256)
// 55.2 / 75.1, 512 (128) 54.0 / 44.8; 16 experts, 8192 tokens (256, half filled) 20.0 / 20.1, 32768 64.5 / 68.5.
// (The selection in the same launch, where a workgroup holds every expert: 27.5 against 24.7 us with 32 experts and 8192 tokens.)
template <typename T>
bool launch_gate_mfma(const void* x, const void* gate_w, const float* gate_bias, float* logits, int S, int H, int E, int opt_mfma, hipStream_t st, hipError_t* err) {
    using G = GateStage<T>;
    if (H % 512 != 0) return false;
    const int et = (E + 15) / 16, etiles = (E + G::ET * 16 - 1) / (G::ET * 16), ttiles = (S + G::TT * 16 - 1) / (G::TT * 16);
    bool use = (etiles * G::ET * 16 * 3 <= E * 4 && (int64_t)ttiles * etiles >= 150) || (et * 16 * 3 <= E * 4 && (int64_t)((S + 15) / 16) * et >= 2048);
    if (opt_mfma != MOE_OPT_AUTO) use = opt_mfma != 0;
    const int64_t tiles = (int64_t)(ttiles + 7) / 8 * 8 * etiles;
    if (!use || tiles > INT32_MAX - 65536) return false;
    *err = hipFuncSetAttribute(reinterpret_cast<const void*>(&gate_mfma_kernel<T>), hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS_BYTES);
    if (*err != hipSuccess) return true;
    gate_mfma_kernel<T><<<(unsigned)std::min<int64_t>(tiles, 256), G::THREADS, G::LDS_BYTES, st>>>((const T*)x, (const T*)gate_w, gate_bias, logits, S, H, E, etiles, (int)tiles);
    *err = hipGetLastError();
    return true;
}

// One wavefront per token.
template <int J>
__global__ __launch_bounds__(256) void topk_kernel(const float* __restrict__ logits, int S, int E, int k, int gate_fn,
                                                   int norm, int32_t* __restrict__ topk_idx,
                                                   float* __restrict__ topk_w) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int t = blockIdx.x * 4 + wave;
    if (t >= S) return;
    topk_one_token<J>(logits + (size_t)t * E, t, E, k, gate_fn, norm, topk_idx, topk_w, lane);
}

// The same for up to 64 experts, sixteen lanes to a token: lane l of a row of sixteen keeps the logits of experts l, l + 16, l + 32 and
// l + 48, so that a candidate travels through four DPP moves instead of four and three lane reads, and a wavefront selects for four tokens
// at a time.  The softmax's sum pairs the experts as the wavefront's butterfly does (e with e + 32, then + 16 in the lane, 8, 4, 2, 1
// between them): the same bits.  16384 tokens x 64 experts, k 6, a token a wavefront / this 17.2 / 8.4 us in a trace
// (profiles/layer_bf16_finegrained_kernel_trace.txt).
struct Cand16 {
    float key, v;
    int i;
};
template <int CTRL>
__device__ __forceinline__ void better16(Cand16& c) {
    Cand16 o;
    o.key = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(c.key), CTRL, 0xF, 0xF, false));
    o.v = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(c.v), CTRL, 0xF, 0xF, false));
    o.i = __builtin_amdgcn_update_dpp(0, c.i, CTRL, 0xF, 0xF, false);
    if (o.key > c.key || (o.key == c.key && o.i < c.i)) c = o;
}
__global__ __launch_bounds__(256) void topk16_kernel(const float* __restrict__ logits, int S, int E, int k, int gate_fn, int norm,
                                                     int32_t* __restrict__ topk_idx, float* __restrict__ topk_w) {
    const int lane = threadIdx.x & 15, t = blockIdx.x * 16 + (threadIdx.x >> 4);
    const bool live = t < S;                       // (a token past the end keeps the lane exchanges company)
    const float* row = logits + (size_t)min(t, S - 1) * E;
    float v[4];
    unsigned avail = 0;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const int e = 16 * m + lane;
        v[m] = 0.0f;
        if (e < E) {
            v[m] = row[e];
            avail |= 1u << m;
        }
    }
    const unsigned valid = avail;
    float my_l = 0.0f, top_l = 0.0f;
    int my_i = 0;
    for (int r = 0; r < k; ++r) {
        Cand16 c{-INFINITY, 0.0f, 0x7FFFFFFF};
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const float key = v[m] != v[m] ? -INFINITY : v[m];
            const int i = 16 * m + lane;
            if (((avail >> m) & 1u) && (key > c.key || (key == c.key && i < c.i))) c = Cand16{key, v[m], i};
        }
        better16<0xB1>(c);                         // quad_perm [1,0,3,2]: lane ^ 1
        better16<0x4E>(c);                         // quad_perm [2,3,0,1]: lane ^ 2
        better16<0x141>(c);                        // row_half_mirror: i <-> 7 - i within 8 lanes
        better16<0x140>(c);                        // row_mirror: i <-> 15 - i
        if ((c.i & 15) == lane) avail &= ~(1u << ((c.i >> 4) & 31));
        if (lane == r) { my_l = c.v; my_i = c.i; }
        if (r == 0) top_l = c.v;
    }
    float p = 0.0f;
    if (gate_fn == MOE_GATE_SOFTMAX) {
        float e[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            e[m] = (valid >> m) & 1u ? expf(v[m] - top_l) : 0.0f;
            asm volatile("" : "+v"(e[m]));         // a value of its own: the library's last product must not melt into the sum
        }
        float part = (e[0] + e[2]) + (e[1] + e[3]);
#pragma unroll
        for (int off = 8; off >= 1; off >>= 1) part = part + __shfl_xor(part, off, 16);
        if (lane < k) p = expf(my_l - top_l) / part;
    } else {
        if (lane < k) p = 1.0f / (1.0f + expf(-my_l));
    }
    if (norm) {
        float sum = p;
#pragma unroll
        for (int off = 8; off >= 1; off >>= 1) sum = sum + __shfl_xor(sum, off, 16);
        p = p / sum;
    }
    if (live && lane < k) {
        topk_idx[(size_t)t * k + lane] = my_i;
        topk_w[(size_t)t * k + lane] = p;
    }
}

// Router statistics for a load-balancing loss.  Block b, wavefront w takes tokens (4b + w) + 4*gridDim.x*i; a lane
// keeps fp64 sums of the gate scores of its experts; wavefront sums meet in LDS in wavefront order and are written as
// per-block partials, so the result does not depend on scheduling.
__global__ __launch_bounds__(256) void router_stats_partial_kernel(const float* __restrict__ logits,
                                                                   const int32_t* __restrict__ topk_idx, int S, int E,
                                                                   int k, int gate_fn, double* __restrict__ part_prob,
                                                                   int32_t* __restrict__ part_cnt) {
    __shared__ double s_sum[4][kMaxExperts];
    __shared__ int s_cnt[kMaxExperts];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    constexpr int J = kMaxExperts / kWave;
    for (int e = threadIdx.x; e < E; e += 256) s_cnt[e] = 0;
    __syncthreads();
    double acc[J];
#pragma unroll
    for (int j = 0; j < J; ++j) acc[j] = 0.0;
    for (int t = blockIdx.x * 4 + wave; t < S; t += 4 * gridDim.x) {
        float v[J];
        float mx = -INFINITY;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int e = j * kWave + lane;
            v[j] = e < E ? logits[(size_t)t * E + e] : -INFINITY;
            mx = fmaxf(mx, v[j]);
        }
        if (gate_fn == MOE_GATE_SOFTMAX) {
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, kWave));
            float part = 0.0f;
#pragma unroll
            for (int j = 0; j < J; ++j) {
                v[j] = j * kWave + lane < E ? expf(v[j] - mx) : 0.0f;
                part = part + v[j];
            }
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) part = part + __shfl_xor(part, off, kWave);
#pragma unroll
            for (int j = 0; j < J; ++j) acc[j] += (double)(v[j] / part);
        } else {
#pragma unroll
            for (int j = 0; j < J; ++j)
                if (j * kWave + lane < E) acc[j] += (double)(1.0f / (1.0f + expf(-v[j])));
        }
        if (lane < k) {
            const int e = topk_idx[(size_t)t * k + lane];
            if ((unsigned)e < (unsigned)E) atomicAdd(&s_cnt[e], 1);   // ids outside [0, E) are counted nowhere
        }
    }
#pragma unroll
    for (int j = 0; j < J; ++j)
        if (j * kWave + lane < E) s_sum[wave][j * kWave + lane] = acc[j];
    __syncthreads();
    for (int e = threadIdx.x; e < E; e += 256) {
        part_prob[(size_t)blockIdx.x * E + e] = ((s_sum[0][e] + s_sum[1][e]) + s_sum[2][e]) + s_sum[3][e];
        part_cnt[(size_t)blockIdx.x * E + e] = s_cnt[e];
    }
}

__global__ __launch_bounds__(512) void router_stats_final_kernel(const double* __restrict__ part_prob,
                                                                 const int32_t* __restrict__ part_cnt, int blocks,
                                                                 int S, int E, int k, float* __restrict__ load,
                                                                 float* __restrict__ mean_prob,
                                                                 float* __restrict__ aux_loss) {
    __shared__ double s_prod[kMaxExperts];
    const int e = threadIdx.x;
    if (e < E) {
        double sum = 0.0;
        long long cnt = 0;
        for (int b = 0; b < blocks; ++b) {
            sum += part_prob[(size_t)b * E + e];
            cnt += part_cnt[(size_t)b * E + e];
        }
        const double mp = sum / (double)S, ld = (double)cnt / ((double)S * (double)k);
        if (mean_prob) mean_prob[e] = (float)mp;
        if (load) load[e] = (float)ld;
        s_prod[e] = mp * ld;
    }
    __syncthreads();
    if (threadIdx.x == 0 && aux_loss) {
        double a = 0.0;
        for (int i = 0; i < E; ++i) a += s_prod[i];
        *aux_loss = (float)((double)E * a);
    }
}

}  // namespace

hipError_t launch_router_stats(const float* logits, const int32_t* topk_idx, int S, int E, int k, int gate_fn,
                               double* part_prob, int32_t* part_cnt, float* load, float* mean_prob, float* aux_loss,
                               hipStream_t st) {
    const int blocks = min(kStatsBlocks, (S + 3) / 4);
    router_stats_partial_kernel<<<blocks, 256, 0, st>>>(logits, topk_idx, S, E, k, gate_fn, part_prob, part_cnt);
    router_stats_final_kernel<<<1, 512, 0, st>>>(part_prob, part_cnt, blocks, S, E, k, load, mean_prob, aux_loss);
    return hipGetLastError();
}

// Logits kernel by shape; *fused (when tk is given) says whether that launch has selected as well.
static hipError_t launch_gate_logits(const void* x, const void* gate_w, const float* gate_bias, float* logits, bool keep_logits,
                                     int S, int H, int E, int act_dtype, const moe_options& opt, const GateTopk* tk, bool* fused,
                                     hipStream_t st) {
    // Many experts on many tokens: the first kernel (token rows in registers, experts streamed) reads least per sum.
    // Everything else -- few experts, or decode-sized batches -- goes to the register-tiled kernel.
    if (act_dtype != MOE_DTYPE_F32) {
        hipError_t e = hipSuccess;
        const bool taken = act_dtype == MOE_DTYPE_FP16
            ? launch_gate_mfma<f16_s>(x, gate_w, gate_bias, logits, S, H, E, opt.gate_mfma, st, &e)
            : launch_gate_mfma<bf16_s>(x, gate_w, gate_bias, logits, S, H, E, opt.gate_mfma, st, &e);
        if (taken) return e;
    }
    bool rows_in_registers = E >= 32 && (int64_t)S * E >= ((int64_t)1 << 19);
    if (opt.gate_kernel != MOE_OPT_AUTO) rows_in_registers = opt.gate_kernel == 1;
    if (rows_in_registers) {
        if (act_dtype == MOE_DTYPE_F32) return launch_gate_typed<float>(x, gate_w, gate_bias, logits, S, H, E, st);
        if (act_dtype == MOE_DTYPE_FP16) return launch_gate_typed<f16_s>(x, gate_w, gate_bias, logits, S, H, E, st);
        return launch_gate_typed<bf16_s>(x, gate_w, gate_bias, logits, S, H, E, st);
    }
    if (act_dtype == MOE_DTYPE_F32) return launch_gate_tiled<float>(x, gate_w, gate_bias, logits, keep_logits, S, H, E, opt.gate_tile, tk, fused, st);
    if (act_dtype == MOE_DTYPE_FP16) return launch_gate_tiled<f16_s>(x, gate_w, gate_bias, logits, keep_logits, S, H, E, opt.gate_tile, tk, fused, st);
    return launch_gate_tiled<bf16_s>(x, gate_w, gate_bias, logits, keep_logits, S, H, E, opt.gate_tile, tk, fused, st);
}

static hipError_t launch_topk(const float* logits, int S, int E, int k, int gate_fn, int norm, int32_t* topk_idx,
                       float* topk_w, hipStream_t st) {
    const unsigned grid = (unsigned)((S + 3) / 4);
    if (E <= 64) topk16_kernel<<<(unsigned)((S + 15) / 16), 256, 0, st>>>(logits, S, E, k, gate_fn, norm, topk_idx, topk_w);
    else if (E <= 128) topk_kernel<2><<<grid, 256, 0, st>>>(logits, S, E, k, gate_fn, norm, topk_idx, topk_w);
    else if (E <= 256) topk_kernel<4><<<grid, 256, 0, st>>>(logits, S, E, k, gate_fn, norm, topk_idx, topk_w);
    else topk_kernel<kMaxExperts / kWave><<<grid, 256, 0, st>>>(logits, S, E, k, gate_fn, norm, topk_idx, topk_w);
    return hipGetLastError();
}

// The router: logits, selection, weights.  One launch where the logits kernel of the shape can hold every expert of a
// token in one workgroup (option gate_fused_topk, on unless 0), else the logits kernel followed by the top-k kernel.
// `logits` is always valid scratch [S, E]; with keep_logits false it is written only when the two-launch form needs it.
hipError_t launch_gate(const void* x, const void* gate_w, const float* gate_bias, float* logits, bool keep_logits, int S,
                       int H, int E, int k, int gate_fn, int norm, int32_t* topk_idx, float* topk_w, int act_dtype,
                       const moe_options& opt, hipStream_t st) {
    const GateTopk tk{topk_idx, topk_w, k, gate_fn, norm};
    bool fused = false;
    const hipError_t e = launch_gate_logits(x, gate_w, gate_bias, logits, keep_logits, S, H, E, act_dtype, opt,
                                            opt.gate_fused_topk == 0 ? nullptr : &tk, &fused, st);
    if (e != hipSuccess || fused) return e;
    return launch_topk(logits, S, E, k, gate_fn, norm, topk_idx, topk_w, st);
}

}  // namespace moe355
