// Building blocks of the backward pass of the expert FFN (the training knob is_training,
// aristos_config.schema.json:20-23, is parsed by the reference and never read; these are this library's).
//
// Everything works on packed expert-major rows as the forward pass lays them out: rows
// [expert_offset[e], expert_offset[e] + expert_count[e]) belong to expert e.
//   * data gradients are grouped (M,K) x (N,K)^T GEMMs with the weight in its K-major view, which a batched transpose
//     produces: dX = dY . W  ==  dY x (W^T)^T.  The forward tile kernels run them unchanged.
//   * weight gradients sum over an expert's rows: dW[e] = dY_e^T . A_e.  Both operands are transposed into buffers whose
//     columns are the packed rows, each expert's window padded with zeros to a multiple of 128 columns, and every
//     expert is then one tile GEMM over its window.
#include <algorithm>

#include <type_traits>

#include "moe_internal.hpp"
#include "act_deriv.hpp"
#include "product_choice.hpp"

namespace moe355 {

bool grouped_hand_ok(int64_t A, int N, int K);
int grouped_gemm_tile_16(int64_t A, int E, int N, int K, int products);
hipError_t launch_grouped_gemm_pair_16(const void* a_rows, const void* w, const void* w1, void* out, void* out1, const int32_t* count,
                                       const int32_t* offset, int tile, int64_t A, int E, int N, int K, bool f16, hipStream_t st);
hipError_t launch_grouped_gemm_kn_pair_16(const void* a_rows, const void* a1_rows, const void* w, const void* w1, void* out, void* out1,
                                          const int32_t* count, const int32_t* offset, bool large, int64_t A, int E, int N, int K, bool f16, hipStream_t st);
hipError_t launch_grouped_gemm_16(const void* a_rows, const void* w, const void* bias, void* out, const int32_t* count,
                                  const int32_t* offset, int tile, int64_t A, int E, int N, int K, int act, bool f16, hipStream_t st);
hipError_t launch_wgrad_16(const void* dyT, const void* aT, void* dw, const int32_t* poff, int E, int N, int K,
                           int64_t ld, bool f16, hipStream_t st);

hipError_t launch_grouped_gemm_kn_16(const void* a_rows, const void* w, const void* u, const void* g_rows, void* out, void* out1,
                                     const int32_t* count, const int32_t* offset, bool large, int64_t A, int E, int N, int K, int hidden_act, bool f16,
                                     hipStream_t st);
hipError_t launch_wgrad_rows_16(const WgradOperands* ops, int n, const int32_t* count, const int32_t* offset, bool large, int E, bool f16, hipStream_t st);
hipError_t launch_grouped_gemm_deriv_16(const void* a_rows, const void* w, const void* u, const void* g_rows, void* du, void* dg,
                                        const int32_t* count, const int32_t* offset, int tile, int64_t A, int E, int N, int K,
                                        int hidden_act, bool f16, hipStream_t st);
hipError_t launch_grouped_gemm_f32(const void* a_rows, const void* w, const void* bias, void* out, const MTile* mtiles,
                                   const int32_t* num_mtiles, int max_mtiles, int N, int K, int act, hipStream_t st);
hipError_t launch_wgrad_f32(const void* dyT, const void* aT, void* dw, const int32_t* poff, int E, int N, int K, int64_t ld,
                            hipStream_t st);
bool grouped_gemm_f32_takes_tile(int64_t A, int N, int K);
hipError_t launch_grouped_gemm_f32_tile(const void* a_rows, const void* w, const void* bias, void* out, const MTile* mtiles,
                                        const int32_t* num_mtiles, int max_mtiles, int N, int K, int act, hipStream_t st);
bool wgrad_f32_takes_tile(int E, int N, int K);
hipError_t launch_wgrad_f32_tile(const void* dyT, const void* aT, void* dw, const int32_t* poff, int E, int N, int K,
                                 int64_t ld, hipStream_t st);

namespace {


// One workgroup: row blocks of `block_m` rows per expert (for the grouped GEMM) and the padded window offsets (for the
// weight gradient).  Either table may be null.
__global__ __launch_bounds__(kMaxExperts) void backward_tables_kernel(const int32_t* __restrict__ count,
                                                                      const int32_t* __restrict__ offset, int E,
                                                                      int block_m, MTile* mtiles, int32_t* num_mtiles,
                                                                      int32_t* poff) {
    __shared__ int s_mt0[kMaxExperts + 1];
    const int e = threadIdx.x;
    if (e == 0) {
        int mt = 0, po = 0;
        for (int i = 0; i < E; ++i) {
            const int n = max(count[i], 0);
            s_mt0[i] = mt;
            mt += (n + block_m - 1) / block_m;
            if (poff) poff[i] = po;
            po += (n + kWindowAlign - 1) / kWindowAlign * kWindowAlign;
        }
        s_mt0[E] = mt;
        if (num_mtiles) *num_mtiles = mt;
        if (poff) poff[E] = po;
    }
    __syncthreads();
    if (e < E && mtiles) {
        const int n = max(count[e], 0), off = offset[e];
        for (int i = 0, mt = s_mt0[e]; mt < s_mt0[e + 1]; ++i, ++mt) {
            MTile t;
            t.expert = e;
            t.row0 = off + i * block_m;
            t.rows = min(block_m, n - i * block_m);
            t.pad = s_mt0[e];        // first row block of this expert (the grouped GEMM orders its tiles by it)
            mtiles[mt] = t;
        }
    }
}

// dst[b][c][r] = src[b][r][c] for 16-bit elements; 64 x 64 tiles through LDS.  grid = (ceil(C/64), ceil(R/64), B).
__global__ __launch_bounds__(256) void transpose16_kernel(const uint16_t* __restrict__ src, uint16_t* __restrict__ dst,
                                                          int64_t R, int64_t C) {
    __shared__ uint16_t tile[64][66];
    const uint16_t* s = src + (size_t)blockIdx.z * R * C;
    uint16_t* d = dst + (size_t)blockIdx.z * R * C;
    const int64_t r0 = (int64_t)blockIdx.y * 64, c0 = (int64_t)blockIdx.x * 64;
    for (int i = threadIdx.x; i < 64 * 64; i += 256) {
        const int r = i >> 6, c = i & 63;
        tile[r][c] = (r0 + r < R && c0 + c < C) ? s[(r0 + r) * C + c0 + c] : (uint16_t)0;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 64 * 64; i += 256) {
        const int c = i >> 6, r = i & 63;
        if (r0 + r < R && c0 + c < C) d[(c0 + c) * R + r0 + r] = tile[r][c];
    }
}
__global__ __launch_bounds__(256) void transpose32_kernel(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst,
                                                          int64_t R, int64_t C) {
    __shared__ uint32_t tile[64][65];
    const uint32_t* s = src + (size_t)blockIdx.z * R * C;
    uint32_t* d = dst + (size_t)blockIdx.z * R * C;
    const int64_t r0 = (int64_t)blockIdx.y * 64, c0 = (int64_t)blockIdx.x * 64;
    for (int i = threadIdx.x; i < 64 * 64; i += 256) {
        const int r = i >> 6, c = i & 63;
        tile[r][c] = (r0 + r < R && c0 + c < C) ? s[(r0 + r) * C + c0 + c] : 0u;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 64 * 64; i += 256) {
        const int c = i >> 6, r = i & 63;
        if (r0 + r < R && c0 + c < C) d[(c0 + c) * R + r0 + r] = tile[r][c];
    }
}

// The same for 16-bit elements when R and C are multiples of 8: every global access is 16 bytes per lane.  A 64 x 64
// tile goes into LDS as rows of 32 dwords + 1 (the odd pitch spreads a column over the banks) and comes out as
// columns, eight 2-byte reads per lane packed into one 16-byte store.
__device__ __forceinline__ void tile64_store_row(uint32_t* tile, int r, int ch, uint4 v) {
    uint32_t* p = tile + r * 33 + ch * 4;
    p[0] = v.x; p[1] = v.y; p[2] = v.z; p[3] = v.w;
}
__device__ __forceinline__ uint4 tile64_load_column(const uint32_t* tile, int col, int row8) {
    const uint16_t* t = reinterpret_cast<const uint16_t*>(tile);
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t lo = t[(row8 * 8 + 2 * j) * 66 + col], hi = t[(row8 * 8 + 2 * j + 1) * 66 + col];
        w[j] = lo | (hi << 16);
    }
    return uint4{w[0], w[1], w[2], w[3]};
}

__global__ __launch_bounds__(256) void transpose16_vec_kernel(const uint16_t* __restrict__ src, uint16_t* __restrict__ dst,
                                                              int64_t R, int64_t C) {
    __shared__ uint32_t tile[64 * 33];
    const uint16_t* s = src + (size_t)blockIdx.z * R * C;
    uint16_t* d = dst + (size_t)blockIdx.z * R * C;
    const int64_t r0 = (int64_t)blockIdx.y * 64, c0 = (int64_t)blockIdx.x * 64;
    const int sub = threadIdx.x >> 3, ch = threadIdx.x & 7;
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
        const int r = sub + 32 * pass;
        uint4 v = {0u, 0u, 0u, 0u};
        if (r0 + r < R && c0 + ch * 8 < C) v = *reinterpret_cast<const uint4*>(s + (r0 + r) * C + c0 + ch * 8);
        tile64_store_row(tile, r, ch, v);
    }
    __syncthreads();
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
        const int c = sub + 32 * pass;
        if (c0 + c < C && r0 + ch * 8 < R)
            *reinterpret_cast<uint4*>(d + (c0 + c) * R + r0 + ch * 8) = tile64_load_column(tile, c, ch);
    }
}

// Packed rows [*, C] -> dst [C, ld]: column poff[e] + s holds row offset[e] + s of expert e (s < count[e]); the rest
// of each window is zero.  A 64-column tile of dst never straddles two windows (they are multiples of 128 wide).
// C is a multiple of 8.  grid = (ld / 64, ceil(C / 64)).
__global__ __launch_bounds__(256) void transpose_rows_padded_kernel(const uint16_t* __restrict__ rows, int C,
                                                                    const int32_t* __restrict__ count,
                                                                    const int32_t* __restrict__ offset,
                                                                    const int32_t* __restrict__ poff, int E, int64_t ld,
                                                                    uint16_t* __restrict__ dst) {
    __shared__ uint32_t tile[64 * 33];
    const int p0 = blockIdx.x * 64;
    if (p0 >= poff[E]) return;                 // behind the last window: never read
    int lo = 0, hi = E - 1;
    while (lo < hi) {                          // last expert whose window starts at or before p0 (empty windows skipped)
        const int mid = (lo + hi + 1) >> 1;
        if (poff[mid] <= p0) lo = mid; else hi = mid - 1;
    }
    const int e = lo, s0 = p0 - poff[e], n = count[e], off = offset[e];
    const int c0 = blockIdx.y * 64;
    const int sub = threadIdx.x >> 3, ch = threadIdx.x & 7;
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
        const int r = sub + 32 * pass;
        uint4 v = {0u, 0u, 0u, 0u};
        if (s0 + r < n && c0 + ch * 8 < C)
            v = *reinterpret_cast<const uint4*>(rows + (size_t)(off + s0 + r) * C + c0 + ch * 8);
        tile64_store_row(tile, r, ch, v);
    }
    __syncthreads();
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
        const int c = sub + 32 * pass;
        if (c0 + c < C)
            *reinterpret_cast<uint4*>(dst + (size_t)(c0 + c) * ld + p0 + ch * 8) = tile64_load_column(tile, c, ch);
    }
}

// The same for 4-byte elements (fp32 layers): any C.  grid = (ld / 64, ceil(C / 64)).
__global__ __launch_bounds__(256) void transpose_rows_padded32_kernel(const uint32_t* __restrict__ rows, int C,
                                                                      const int32_t* __restrict__ count,
                                                                      const int32_t* __restrict__ offset,
                                                                      const int32_t* __restrict__ poff, int E, int64_t ld,
                                                                      uint32_t* __restrict__ dst) {
    __shared__ uint32_t tile[64][65];
    const int p0 = blockIdx.x * 64;
    if (p0 >= poff[E]) return;                 // behind the last window: never read
    int lo = 0, hi = E - 1;
    while (lo < hi) {                          // last expert whose window starts at or before p0 (empty windows skipped)
        const int mid = (lo + hi + 1) >> 1;
        if (poff[mid] <= p0) lo = mid; else hi = mid - 1;
    }
    const int e = lo, s0 = p0 - poff[e], n = count[e], off = offset[e];
    const int c0 = blockIdx.y * 64;
    for (int i = threadIdx.x; i < 64 * 64; i += 256) {
        const int r = i >> 6, c = i & 63;
        tile[r][c] = (s0 + r < n && c0 + c < C) ? rows[(size_t)(off + s0 + r) * C + c0 + c] : 0u;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 64 * 64; i += 256) {
        const int c = i >> 6, r = i & 63;
        if (c0 + c < C) dst[(size_t)(c0 + c) * ld + p0 + r] = tile[r][c];
    }
}

// ---- elementwise and reduction steps of a backward pass ----
struct f32_s {};
template <class T> struct RawOf { typedef uint16_t type; };
template <> struct RawOf<f32_s> { typedef float type; };
template <class T16> __device__ __forceinline__ float ld16(const typename RawOf<T16>::type* p, size_t i);
template <> __device__ __forceinline__ float ld16<bf16_s>(const uint16_t* p, size_t i) { return __uint_as_float((uint32_t)p[i] << 16); }
template <> __device__ __forceinline__ float ld16<f16_s>(const uint16_t* p, size_t i) { return (float)__builtin_bit_cast(_Float16, p[i]); }
template <> __device__ __forceinline__ float ld16<f32_s>(const float* p, size_t i) { return p[i]; }
template <class T16> __device__ __forceinline__ typename RawOf<T16>::type st16(float v);
template <> __device__ __forceinline__ uint16_t st16<bf16_s>(float v) {
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
    const f32x2_t x = {v, 0.0f};
    return (uint16_t)(__builtin_bit_cast(uint32_t, __builtin_convertvector(x, bf16x2_t)) & 0xFFFFu);
}
template <> __device__ __forceinline__ uint16_t st16<f16_s>(float v) { return __builtin_bit_cast(uint16_t, (_Float16)v); }
template <> __device__ __forceinline__ float st16<f32_s>(float v) { return v; }

// du = dh * act'(u); SwiGLU (h = silu(g) u): du = dh silu(g), dg = dh u s (1 + g (1 - s)), s = sigmoid(g).
// fp32 layers use the library functions; 16-bit layers the forms of act_deriv.hpp, which the fused data gradient's
// epilogue inlines as well (same bits on both paths).
template <class T16>
__device__ __forceinline__ void act_backward_one(float d, float uv, float gv, int act, float& a, float& b) {
    constexpr bool kF32 = std::is_same<T16, f32_s>::value;
    b = 0.0f;
    if (act == MOE_ACT_SWIGLU) {
        if constexpr (kF32) {
            const float sg = 1.0f / (1.0f + expf(-gv));
            a = d * (gv * sg);
            b = d * uv * (sg * (1.0f + gv * (1.0f - sg)));
        } else {
            dswiglu16(d, uv, gv, a, b);
        }
    } else if (act == MOE_ACT_GELU) {
        if constexpr (kF32) {
            const float cdf = 0.5f * (1.0f + erff(uv * 0.70710678118654752440f));
            const float pdf = 0.39894228040143267794f * expf(-0.5f * uv * uv);
            a = d * (cdf + uv * pdf);
        } else {
            a = dgelu16(d, uv);
        }
    } else {
        a = drelu16(d, uv);
    }
}

constexpr int kRowsPass = 2;           // 16-byte pieces a thread of the pass below has in flight of every operand
// 16 bytes of every operand per thread and step (8 or 4 elements): the pass is a stream over five arrays at most and
// has nothing else to wait for.  n is a multiple of the intermediate size, which is a multiple of 64; all pointers
// 16-byte aligned (the launcher checks both).
template <class T16, class RAW = typename RawOf<T16>::type>
__global__ __launch_bounds__(256) void act_backward_kernel(const RAW* __restrict__ dh, const RAW* __restrict__ u,
                                                           const RAW* __restrict__ g, size_t n, int act,
                                                           RAW* __restrict__ du, RAW* __restrict__ dg) {
    constexpr int VEC = 16 / (int)sizeof(RAW);
    union Pack { uint4 q; RAW e[VEC]; };
    const size_t nv = n / VEC, id = (size_t)blockIdx.x * 256 + threadIdx.x;
    const bool gated = act == MOE_ACT_SWIGLU;
    for (size_t i = id; i < nv; i += (size_t)gridDim.x * 256) {
        Pack d, uu, gg, oa, ob;
        d.q = reinterpret_cast<const uint4*>(dh)[i];
        uu.q = reinterpret_cast<const uint4*>(u)[i];
        gg.q = gated ? reinterpret_cast<const uint4*>(g)[i] : uint4{0u, 0u, 0u, 0u};
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
            float a, b;
            act_backward_one<T16>(ld16<T16>(d.e, k), ld16<T16>(uu.e, k), ld16<T16>(gg.e, k), act, a, b);
            oa.e[k] = st16<T16>(a);
            ob.e[k] = st16<T16>(b);
        }
        reinterpret_cast<uint4*>(du)[i] = oa.q;
        if (gated) reinterpret_cast<uint4*>(dg)[i] = ob.q;
    }
}

// The same in place behind a data gradient of the rows that belong to an expert: du holds dh and becomes du.  Rows of no expert are
// neither read nor written.  Behind the 256-row tiles this pass is faster than their epilogue with the derivative in it, whose
// arithmetic (14 us a tile) the one wavefront of a SIMD hides behind nothing; behind the 128-row tile, two thirds of whose tasks share a
// round with others, it is not.  SwiGLU, bf16, us, epilogue / pass: 256-row blocks, 16 experts of 2048 x 2048, 512 rows each 128 / 117; 4 of
// 2048 x 2560, 4096 rows 244 / 221; 128-row blocks, 8 of 1280 x 1664, 250 rows 30 / 30; 16 of 1152 x 1920, 175 rows 32 / 34; 4 of
// 1024 x 2560, 750 rows 30 / 36.
template <class T16>
__global__ __launch_bounds__(256) void act_backward_rows_kernel(const uint16_t* __restrict__ u, const uint16_t* __restrict__ g,
                                                                const int32_t* __restrict__ count, const int32_t* __restrict__ offset,
                                                                int E, int64_t A, int N, int act, uint16_t* du, uint16_t* __restrict__ dg) {
    union Pack { uint4 q; uint16_t e[8]; };
    const int64_t kept = offset[E - 1] + count[E - 1];
    const size_t nv = (size_t)(kept < A ? kept : A) * N / 8;
    const bool gated = act == MOE_ACT_SWIGLU;
    const size_t i0 = (size_t)blockIdx.x * (256 * kRowsPass) + threadIdx.x;
    Pack d[kRowsPass], uu[kRowsPass], gg[kRowsPass];
#pragma unroll
    for (int p = 0; p < kRowsPass; ++p) {
        const size_t i = i0 + p * 256;
        if (i >= nv) break;
        d[p].q = reinterpret_cast<const uint4*>(du)[i];
        uu[p].q = reinterpret_cast<const uint4*>(u)[i];
        gg[p].q = gated ? reinterpret_cast<const uint4*>(g)[i] : uint4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int p = 0; p < kRowsPass; ++p) {
        const size_t i = i0 + p * 256;
        if (i >= nv) break;
        Pack oa, ob;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            float a, b;
            act_backward_one<T16>(ld16<T16>(d[p].e, k), ld16<T16>(uu[p].e, k), ld16<T16>(gg[p].e, k), act, a, b);
            oa.e[k] = st16<T16>(a);
            ob.e[k] = st16<T16>(b);
        }
        reinterpret_cast<uint4*>(du)[i] = oa.q;
        if (gated) reinterpret_cast<uint4*>(dg)[i] = ob.q;
    }
}

// The same one element at a time, for operands that are not 16-byte aligned.
template <class T16, class RAW = typename RawOf<T16>::type>
__global__ __launch_bounds__(256) void act_backward_unaligned_kernel(const RAW* __restrict__ dh, const RAW* __restrict__ u,
                                                                     const RAW* __restrict__ g, size_t n, int act,
                                                                     RAW* __restrict__ du, RAW* __restrict__ dg) {
    const bool gated = act == MOE_ACT_SWIGLU;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        float a, b;
        act_backward_one<T16>(ld16<T16>(dh, i), ld16<T16>(u, i), gated ? ld16<T16>(g, i) : 0.0f, act, a, b);
        du[i] = st16<T16>(a);
        if (gated) dg[i] = st16<T16>(b);
    }
}

// db[e, n] = sum over expert e's rows, ascending, of dy[r, n]: one thread per column, so the order is fixed.
// grid = (ceil(N / 256), E).
template <class T16, class RAW = typename RawOf<T16>::type>
__global__ __launch_bounds__(256) void bias_grad_kernel(const RAW* __restrict__ dy, const int32_t* __restrict__ count,
                                                        const int32_t* __restrict__ offset, int N, RAW* __restrict__ db) {
    const int n = blockIdx.x * 256 + threadIdx.x, e = blockIdx.y;
    if (n >= N) return;
    const int r0 = offset[e], r1 = r0 + max(count[e], 0);
    float acc = 0.0f;
    for (int r = r0; r < r1; ++r) acc = acc + ld16<T16>(dy, (size_t)r * N + n);
    db[(size_t)e * N + n] = st16<T16>(acc);
}

// Where the combine's adjoint leaves the gradient of the router's logits (null dl: not asked for).
struct RouterGrad {
    const int32_t* topk_idx;     // [S, k]
    const float* logits;         // [S, E], read where the gate is a normalised sigmoid only
    float* dl;                   // [S, k]: of the chosen experts' logits (those of the others are zero)
    float* dl_dense;             // [S, ld]: the same as rows over the experts, zeros elsewhere
    int32_t* row_of;             // [S]: a packed row that holds the token, -1 where all of its pairs were dropped (its dl are zeros)
    int E, ld, gate_fn, norm;
};
// The adjoint of the gate weights of one token (one wavefront; lane j < k holds dw of rank j), in fp32:
//   softmax, normalised over the chosen: w = softmax of the chosen logits,  dl_j = w_j (dw_j - sum_m w_m dw_m);
//   sigmoid: dl_j = s_j (1 - s_j) dw_j, s = w;  normalised: ds_j = (dw_j - sum_m w_m dw_m) / sum_m s_m, dl_j = s_j (1 - s_j) ds_j.
__device__ __forceinline__ void router_grad_token(const RouterGrad& r, const float* __restrict__ topk_w, float dw, int row, int t, int k) {
    const int lane = threadIdx.x & 63;
    if (lane == 0) r.row_of[t] = row;
    const bool have = lane < k;
    const int e = have ? r.topk_idx[(size_t)t * k + lane] : -1;
    const float w = have ? topk_w[(size_t)t * k + lane] : 0.0f;
    auto sum = [](float v) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
        return v;
    };
    float g = dw;
    if (r.norm) g -= sum(w * dw);
    float dl;
    if (r.gate_fn == MOE_GATE_SOFTMAX) {
        dl = w * g;
    } else {
        float s = w;
        if (r.norm) {
            s = have ? 1.0f / (1.0f + expf(-r.logits[(size_t)t * r.E + e])) : 0.0f;
            g /= sum(s);
        }
        dl = s * (1.0f - s) * g;
    }
    if (have) r.dl[(size_t)t * k + lane] = dl;
    for (int c = lane; c - lane < r.ld; c += 64) {       // every lane takes every turn: the shuffles read all of them
        float v = 0.0f;
        for (int j = 0; j < k; ++j) {
            const float d = __shfl(dl, j, 64);
            if (__shfl(e, j, 64) == c) v = d;
        }
        if (c < r.ld) r.dl_dense[(size_t)t * r.ld + c] = v;
    }
}

// The router's weight gradient, dgate_w[e, :] = sum over tokens of dl[t, e] x[t, :], in fp32: a share of the tokens a wavefront,
// 256 columns x 16 experts of sums in its registers, the coefficients as scalars; the four wavefronts' sums meet in LDS and the
// workgroups' in gate_wgrad_sum_kernel, both in a fixed order.  grid = (columns / 256, shares, experts / 16).  row_of: null, or x are the
// packed rows, and a token is read from the one that row_of names.
constexpr int kGateShareMax = 64;      // partial sums of E * H * 4 bytes each: never more than the transposed operands the scratch is sized for
template <class T16, class RAW = typename RawOf<T16>::type>
__global__ __launch_bounds__(256) void gate_wgrad_kernel(const RAW* __restrict__ x, const int32_t* __restrict__ row_of, const float* __restrict__ dl, int S, int H, int E, int ld, float* __restrict__ part) {
    __shared__ float red[4][64][64];   // [wavefront][expert * 4 + column of the lane][lane]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = blockIdx.x * 256 + 4 * lane, e0 = blockIdx.z * 16;
    const int shares = gridDim.y * 4, per = (S + shares - 1) / shares;
    const int t0 = (blockIdx.y * 4 + wave) * per, t1 = min(S, t0 + per);
    float acc[16][4];
#pragma unroll
    for (int e = 0; e < 16; ++e)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[e][v] = 0.0f;
    const int c = col < H ? col : 0;
    struct alignas(4 * sizeof(RAW)) Four { RAW e[4]; };
#pragma unroll 4
    for (int t = t0; t < t1; ++t) {
        const int row = row_of ? row_of[t] : t;
        Four q = *reinterpret_cast<const Four*>(x + (size_t)max(row, 0) * H + c);
        if (row < 0) q = Four{};               // no packed row: whatever row 0 holds, infinities too, takes no part
        const float* d = dl + (size_t)t * ld + e0;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const float w = d[e];
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[e][v] = fmaf(w, ld16<T16>(q.e, v), acc[e][v]);
        }
    }
#pragma unroll
    for (int e = 0; e < 16; ++e)
#pragma unroll
        for (int v = 0; v < 4; ++v) red[wave][e * 4 + v][lane] = acc[e][v];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {              // this wavefront: experts 4 wave .. + 3
        const int e = 4 * wave + i;
        float o[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) o[v] = (red[0][e * 4 + v][lane] + red[1][e * 4 + v][lane]) + (red[2][e * 4 + v][lane] + red[3][e * 4 + v][lane]);
        if (col < H && e0 + e < E) *reinterpret_cast<float4*>(part + ((size_t)blockIdx.y * E + e0 + e) * H + col) = float4{o[0], o[1], o[2], o[3]};
    }
}
template <class T16, class RAW = typename RawOf<T16>::type>
__global__ __launch_bounds__(256) void gate_wgrad_sum_kernel(const float* __restrict__ part, int shares, int n, RAW* __restrict__ dw) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    float sum = 0.0f;
#pragma unroll 8
    for (int s = 0; s < shares; ++s) sum = sum + part[(size_t)s * n + i];
    dw[i] = st16<T16>(sum);
}

// dy[row(t,r), :] = w[t,r] * dout[t, :]; dw[t,r] = <dout[t, :], y[row(t,r), :]>, one wavefront per token, four tokens per
// workgroup.  Bound by memory (dout and y in, dy out): 16 bytes per lane and operand, the rows of four ranks in flight
// beside one load of dout, and the dot products fold across the wavefront without LDS or a barrier.  8192 tokens x 2
// ranks x 2048 columns in bf16 would be 168 MB; H is a multiple of 64 and every operand 16-byte aligned (launcher).
template <class T16, class RAW = typename RawOf<T16>::type>
__global__ __launch_bounds__(256) void combine_backward_kernel(const RAW* __restrict__ dout, const RAW* __restrict__ y,
                                                               const int32_t* __restrict__ pair_row,
                                                               const float* __restrict__ topk_w, int S, int k, int H,
                                                               RAW* __restrict__ dy, float* __restrict__ dw, RouterGrad router) {
    constexpr int VEC = 16 / (int)sizeof(RAW);
    union Pack { uint4 q; RAW e[VEC]; };
    const int lane = threadIdx.x & 63, t = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= S) return;
    float mine = 0.0f;                 // lane j: dw[t, j]
    int held = -1;                     // the token's first packed row
    for (int r0 = 0; r0 < k; r0 += 4) {
        int row[4];
        float w[4], acc[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            row[j] = r0 + j < k ? __builtin_amdgcn_readfirstlane(pair_row[(size_t)t * k + r0 + j]) : -1;
            w[j] = row[j] >= 0 ? topk_w[(size_t)t * k + r0 + j] : 0.0f;
            acc[j] = 0.0f;
        }
        for (int c = lane * VEC; c < H; c += 64 * VEC) {
            Pack d, v[4], o;
            d.q = *reinterpret_cast<const uint4*>(dout + (size_t)t * H + c);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (row[j] >= 0) v[j].q = *reinterpret_cast<const uint4*>(y + (size_t)row[j] * H + c);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (row[j] < 0) continue;
#pragma unroll
                for (int i = 0; i < VEC; ++i) {
                    const float di = ld16<T16>(d.e, i);
                    o.e[i] = st16<T16>(settled(w[j] * di));
                    acc[j] = fmaf(di, ld16<T16>(v[j].e, i), acc[j]);
                }
                *reinterpret_cast<uint4*>(dy + (size_t)row[j] * H + c) = o.q;
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) acc[j] += __shfl_xor(acc[j], off, 64);
            if (row[j] < 0) acc[j] = 0.0f;
            else if (held < 0) held = row[j];
            if (lane == r0 + j) mine = acc[j];
            if (dw && lane == 0 && r0 + j < k) dw[(size_t)t * k + r0 + j] = acc[j];
        }
    }
    if (router.dl) router_grad_token(router, topk_w, mine, held, t, k);
}

// The same one element at a time, for operands that are not 16-byte aligned: one workgroup per token.
template <class T16, class RAW = typename RawOf<T16>::type>
__global__ __launch_bounds__(256) void combine_backward_unaligned_kernel(const RAW* __restrict__ dout, const RAW* __restrict__ y,
                                                               const int32_t* __restrict__ pair_row,
                                                               const float* __restrict__ topk_w, int k, int H,
                                                               RAW* __restrict__ dy, float* __restrict__ dw) {
    __shared__ float part[4];
    const int t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int r = 0; r < k; ++r) {
        const int row = pair_row[(size_t)t * k + r];
        float acc = 0.0f;
        if (row >= 0) {
            const float w = topk_w[(size_t)t * k + r];
            for (int j = threadIdx.x; j < H; j += 256) {
                const float d = ld16<T16>(dout, (size_t)t * H + j);
                dy[(size_t)row * H + j] = st16<T16>(settled(w * d));
                acc = fmaf(d, ld16<T16>(y, (size_t)row * H + j), acc);
            }
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
        __syncthreads();                       // part may still be read for the previous rank
        if (lane == 0) part[wave] = acc;
        __syncthreads();
        if (threadIdx.x == 0) dw[(size_t)t * k + r] = row >= 0 ? (part[0] + part[1]) + (part[2] + part[3]) : 0.0f;
    }
}

// h = act(u) (SwiGLU: silu(g) * u) over the packed rows that belong to an expert; what lies behind them is not touched.
// The library's erff / expf and a true division, in fp32, for every type: what a training step computed as torch expressions.
// (The tiles' silu16 and gelu16 are good to 5e-7 absolute; in fp16 GELU's tail that is 1.2 instead of 1.0 units of the last place.)
__device__ __forceinline__ float act_forward_one(float u, float g, int act) {
    if (act == MOE_ACT_SWIGLU) return settled(g / (1.0f + expf(-g)) * u);
    if (act == MOE_ACT_GELU) return settled(0.5f * u * (1.0f + erff(u * 0.70710678118654752440f)));
    return u < 0.0f ? 0.0f : u;      // a NaN stays a NaN
}

// A stream over two or three arrays, 16 bytes per thread and operand.  8192 rows x 2048 columns of GELU in bf16 (67 MB):
// the widening copy, the activation and the narrowing copy of a torch expression took 16 + 22 + 15 us.
template <class T16, class RAW = typename RawOf<T16>::type>
__global__ __launch_bounds__(256) void act_forward_kernel(const RAW* __restrict__ u, const RAW* __restrict__ g,
                                                          const int32_t* __restrict__ count,
                                                          const int32_t* __restrict__ offset, int E, int64_t A, int I, int act,
                                                          RAW* __restrict__ h) {
    constexpr int VEC = 16 / (int)sizeof(RAW);
    union Pack { uint4 q; RAW e[VEC]; };
    const int64_t kept = offset[E - 1] + count[E - 1];
    const size_t nv = (size_t)(kept < A ? kept : A) * I / VEC;
    const bool gated = act == MOE_ACT_SWIGLU;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < nv; i += (size_t)gridDim.x * 256) {
        Pack uu, gg, o;
        uu.q = reinterpret_cast<const uint4*>(u)[i];
        gg.q = gated ? reinterpret_cast<const uint4*>(g)[i] : uint4{0u, 0u, 0u, 0u};
#pragma unroll
        for (int k = 0; k < VEC; ++k) o.e[k] = st16<T16>(act_forward_one(ld16<T16>(uu.e, k), ld16<T16>(gg.e, k), act));
        reinterpret_cast<uint4*>(h)[i] = o.q;
    }
}

// rows[r, :] = x[token_indices[r], :] for the packed rows that belong to an expert: the dispatch as a pass of its own (a
// training step keeps the rows for the weight gradients).  One wavefront per row, 16 bytes per lane.
__global__ __launch_bounds__(256) void dispatch_rows_kernel(const uint4* __restrict__ x,
                                                            const int32_t* __restrict__ token_indices, int64_t A, int row_vec,
                                                            int S, uint4* __restrict__ rows) {
    const int lane = threadIdx.x & 63;
    const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= A) return;
    const int t = __builtin_amdgcn_readfirstlane(token_indices[r]);
    if ((unsigned)t >= (unsigned)S) return;      // behind the last kept row
    for (int c = lane; c < row_vec; c += 64) rows[r * row_vec + c] = x[(int64_t)t * row_vec + c];
}

// dx[t, :] = sum over ranks r, ascending, of a[pair_row[t,r], :] + b[pair_row[t,r], :] (b may be null), and, with dl, behind
// them of dl[t,r] gate_w[topk_idx[t,r], :], in fp32 and rounded once: the adjoint of the dispatch for one or two row gradients.
// Bound by latency more than by its bytes: what a piece reads hangs on its token's ranks, two trips to memory behind each other.  So a
// wavefront takes one piece (64 x 16 bytes) of a token, not a token, and asks for the rows of four ranks and the router's weight
// rows of the same ranks before it adds anything.  A wavefront per token, piece after piece, the router's ranks one after the other / this:
// us, bf16, with the router's share: 3000 tokens x 4, rows of 2048, two gradients 24.1 / 21.8; 16384 x 6 225 / 183; 8192 x 2, rows of 4096
// 112 / 70 (a copy of the same bytes 18, 139, 53); 4096 x 2, one gradient 13.4 / 13.7.  (The combine's adjoint with a token's pieces over
// four wavefronts: 198 / 169 and 91 / 70 for the two large ones, but 20.3 / 21.1 and 16.3 / 18.4 for the others: not done.)
template <class T16, class RAW = typename RawOf<T16>::type>
__global__ __launch_bounds__(256) void dispatch_backward_kernel(const RAW* __restrict__ a, const RAW* __restrict__ b,
                                                                const int32_t* __restrict__ pair_row, int S, int k, int H, int pieces,
                                                                RAW* __restrict__ dx, const int32_t* __restrict__ topk_idx,
                                                                const float* __restrict__ dl, const RAW* __restrict__ gate_w) {
    constexpr int VEC = 16 / (int)sizeof(RAW);
    union Pack { uint4 q; RAW e[VEC]; };
    const int64_t id = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t = (int)(id / pieces), c = ((int)(id - (int64_t)t * pieces) * 64 + (threadIdx.x & 63)) * VEC;
    if (t >= S || c >= H) return;
    const int32_t* rows = pair_row + (size_t)t * k;
    const int32_t* experts = topk_idx + (size_t)t * k;
    const float* d = dl + (size_t)t * k;
    Pack w[4];
    float scale[4];
    auto router_rows = [&](int r0) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (r0 + j >= k) continue;
            scale[j] = d[r0 + j];
            w[j].q = *reinterpret_cast<const uint4*>(gate_w + (size_t)__builtin_amdgcn_readfirstlane(experts[r0 + j]) * H + c);
        }
    };
    if (dl) router_rows(0);
    float acc[VEC];
#pragma unroll
    for (int i = 0; i < VEC; ++i) acc[i] = 0.0f;
    for (int r0 = 0; r0 < k; r0 += 4) {
        int row[4];
        Pack va[4], vb[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            row[j] = r0 + j < k ? __builtin_amdgcn_readfirstlane(rows[r0 + j]) : -1;
            if (row[j] < 0) continue;
            va[j].q = *reinterpret_cast<const uint4*>(a + (size_t)row[j] * H + c);
            if (b) vb[j].q = *reinterpret_cast<const uint4*>(b + (size_t)row[j] * H + c);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (row[j] < 0) continue;
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                acc[i] = acc[i] + ld16<T16>(va[j].e, i);
                if (b) acc[i] = acc[i] + ld16<T16>(vb[j].e, i);
            }
        }
    }
    if (dl) {
        for (int r0 = 0; r0 < k; r0 += 4) {
            if (r0) router_rows(r0);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (r0 + j >= k) continue;
#pragma unroll
                for (int i = 0; i < VEC; ++i) acc[i] = fmaf(scale[j], ld16<T16>(w[j].e, i), acc[i]);
            }
        }
    }
    Pack o;
#pragma unroll
    for (int i = 0; i < VEC; ++i) o.e[i] = st16<T16>(acc[i]);
    *reinterpret_cast<uint4*>(dx + (size_t)t * H + c) = o.q;
}

size_t align256(size_t v) { return (v + 255) / 256 * 256; }

}  // namespace


size_t backward_scratch_bytes(int64_t A, int E, int H, int I, int elem_bytes) {
    const size_t tables = align256(sizeof(int32_t)) + align256((size_t)(A / 64 + E + 1) * sizeof(MTile)) + align256((size_t)(E + 1) * 4);
    const size_t operands = align256((size_t)H * wgrad_ld(A, E) * elem_bytes) + align256((size_t)I * wgrad_ld(A, E) * elem_bytes);
    return tables + operands;
}

hipError_t launch_transpose(const void* src, void* dst, int64_t batch, int64_t rows, int64_t cols, int elem_bytes,
                            hipStream_t st) {
    if (batch < 1 || rows < 1 || cols < 1) return hipSuccess;
    const dim3 grid((unsigned)((cols + 63) / 64), (unsigned)((rows + 63) / 64), (unsigned)batch);
    if (elem_bytes == 2 && rows % 8 == 0 && cols % 8 == 0 && ((uintptr_t)src % 16 == 0) && ((uintptr_t)dst % 16 == 0))
        transpose16_vec_kernel<<<grid, 256, 0, st>>>((const uint16_t*)src, (uint16_t*)dst, rows, cols);
    else if (elem_bytes == 2) transpose16_kernel<<<grid, 256, 0, st>>>((const uint16_t*)src, (uint16_t*)dst, rows, cols);
    else transpose32_kernel<<<grid, 256, 0, st>>>((const uint32_t*)src, (uint32_t*)dst, rows, cols);
    return hipGetLastError();
}

namespace {
// The table region at the head of the scratch buffer: the number of row blocks, the row blocks (64 rows is the
// smallest block any kernel here uses), the window offsets.
struct ScratchTables {
    int32_t* num_mtiles;
    MTile* mtiles;
    int32_t* poff;
    char* operands;
};
ScratchTables scratch_tables(void* scratch, int64_t A, int E) {
    char* s = static_cast<char*>(scratch);
    ScratchTables t;
    t.num_mtiles = reinterpret_cast<int32_t*>(s);
    t.mtiles = reinterpret_cast<MTile*>(s + align256(sizeof(int32_t)));
    const size_t tables = align256(sizeof(int32_t)) + align256((size_t)(A / 64 + E + 1) * sizeof(MTile));
    t.poff = reinterpret_cast<int32_t*>(s + tables);
    t.operands = s + tables + align256((size_t)(E + 1) * 4);
    return t;
}
}  // namespace

// Tile of 16-bit products: 1: 256 x 256, 2: 128 x 256, 0: 128 x 128.
static int product_tile(int64_t A, int E, int N, int K, int products, const moe_options& opt) {
    const int v = opt.grouped_tile;
    if (v == 0) return 0;
    return (v == 1 || v == 2) && grouped_hand_ok(A, N, K) ? v : grouped_gemm_tile_16(A, E, N, K, products);
}

// out_rows[r,:] = act(a_rows[r,:] . w[e(r)]^T + bias[e(r)]); scratch: the row-block table of an fp32 product (16-bit ones
// find their row blocks themselves).
// dtype: the storage type of every operand (MOE_DTYPE_F32, _BF16 or _FP16).
hipError_t launch_expert_gemm(const void* a_rows, const void* w, const void* bias, const int32_t* count,
                              const int32_t* offset, int64_t A, int E, int N, int K, int act, int dtype,
                              const moe_options& opt, void* out_rows, void* scratch, hipStream_t st) {
    if (dtype == MOE_DTYPE_F32) {
        const ScratchTables t = scratch_tables(scratch, A, E);
        bool mfma = grouped_gemm_f32_takes_tile(A, N, K);
        if (opt.f32_tile == 0) mfma = false;   // option: keep the vector-ALU kernel
        const int block_m = mfma ? 128 : 64;
        const int max_mtiles = (int)(A / block_m + E);
        backward_tables_kernel<<<1, kMaxExperts, 0, st>>>(count, offset, E, block_m, t.mtiles, t.num_mtiles, nullptr);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        return (mfma ? launch_grouped_gemm_f32_tile : launch_grouped_gemm_f32)(a_rows, w, bias, out_rows, t.mtiles,
                                                                               t.num_mtiles, max_mtiles, N, K, act, st);
    }
    const int tile = product_tile(A, E, N, K, 1, opt);
    return launch_grouped_gemm_16(a_rows, w, bias, out_rows, count, offset, tile, A, E, N, K, act, dtype == MOE_DTYPE_FP16, st);
}

// out0 = a_rows . w0[e]^T and out1 = a_rows . w1[e]^T: one launch on the hand-ordered tiles, else two calls.
hipError_t launch_expert_gemm_pair(const void* a_rows, const void* w0, const void* w1, const int32_t* count, const int32_t* offset, int64_t A,
                                   int E, int N, int K, int dtype, const moe_options& opt, void* out0, void* out1, void* scratch, hipStream_t st) {
    const int tile = dtype == MOE_DTYPE_F32 ? 0 : product_tile(A, E, N, K, 2, opt);
    if (tile) return launch_grouped_gemm_pair_16(a_rows, w0, w1, out0, out1, count, offset, tile, A, E, N, K, dtype == MOE_DTYPE_FP16, st);
    const hipError_t e = launch_expert_gemm(a_rows, w0, nullptr, count, offset, A, E, N, K, MOE_ACT_NONE, dtype, opt, out0, scratch, st);
    if (e != hipSuccess) return e;
    return launch_expert_gemm(a_rows, w1, nullptr, count, offset, A, E, N, K, MOE_ACT_NONE, dtype, opt, out1, scratch, st);
}

// The tile the fused data gradient (product + activation derivative) runs on: 1 or 2 (the hand-ordered tiles), or 0 where
// there is none: option grouped_tile = 0 (the 128 x 128 tile has no such epilogue), operands of 4 GiB and more, and ragged
// dimensions.  The tiles themselves take those; what moe_expert_gemm_act_backward_supported answers for them, and the
// two-call chain behind it, is from before they did.
int expert_gemm_dact_tile(int64_t A, int E, int N, int K, int dtype, const moe_options& opt) {
    if (dtype != MOE_DTYPE_BF16 && dtype != MOE_DTYPE_FP16) return 0;
    const bool hand_ok = N % 256 == 0 && K % 128 == 0 && grouped_hand_ok(A, N, K);
    int tile = hand_ok ? grouped_gemm_tile_16(A, E, N, K, 1) : 0;
    if (opt.grouped_tile != MOE_OPT_AUTO) {
        const int v = opt.grouped_tile;
        if ((v == 1 || v == 2) && hand_ok) tile = v;
        if (v == 0) tile = 0;
    }
    return tile;
}

// du_rows = (dy_rows . w[e(r)]^T) * act'(u_rows) (and dg_rows for SwiGLU): launch_expert_gemm with act NONE and
// launch_act_backward in one kernel; the product is rounded to the storage type before the derivative, as the two-call
// chain does when it stores dh, so both give the same bits.  16-bit layers on the hand-ordered tiles only.
hipError_t launch_expert_gemm_dact(const void* dy_rows, const void* w, const void* u_rows, const void* g_rows,
                                   const int32_t* count, const int32_t* offset, int64_t A, int E, int N, int K, int hidden_act,
                                   int dtype, const moe_options& opt, void* du_rows, void* dg_rows, void* scratch,
                                   hipStream_t st) {
    const int tile = expert_gemm_dact_tile(A, E, N, K, dtype, opt);
    if (tile == 0) return hipErrorNotSupported;
    return launch_grouped_gemm_deriv_16(dy_rows, w, u_rows, g_rows, du_rows, dg_rows, count, offset, tile, A, E, N, K, hidden_act,
                                        dtype == MOE_DTYPE_FP16, st);
}

static bool overlap(const void* a, const void* b, int64_t bytes) {
    return a && b && (uintptr_t)a < (uintptr_t)b + bytes && (uintptr_t)b < (uintptr_t)a + bytes;
}
// out_rows[r,:] = a_rows[r,:] . w[e(r)] with w [E, K, N] as the other direction stores it, and with u_rows the derivative behind it
// (launch_expert_gemm_dact): no transposed copy of the weight.  16-bit layers.
int expert_gemm_kn_supported(int64_t A, int E, int N, int K, int dtype, const moe_options& opt) {
    if (dtype == MOE_DTYPE_F32 || !stored_operands_ok(A, N, K)) return 0;
    return opt.grouped_tile == MOE_OPT_AUTO && stored_operands_ok(A, N, K) ? 2 : 1;
}
hipError_t launch_expert_gemm_kn(const void* a_rows, const void* w, const void* u_rows, const void* g_rows, const int32_t* count,
                                 const int32_t* offset, int64_t A, int E, int N, int K, int hidden_act, int dtype, void* out_rows, void* out1_rows,
                                 hipStream_t st) {
    if (dtype == MOE_DTYPE_F32 || !stored_operands_ok(A, N, K)) return hipErrorNotSupported;
    const bool f16 = dtype == MOE_DTYPE_FP16, large = grouped_kn_large(A, E, N, K);
    // (results on top of the saved projections: the epilogue reads those before it writes)
    const bool in_place = u_rows && (overlap(out_rows, u_rows, A * N * 2) || overlap(out_rows, g_rows, A * N * 2) || overlap(out1_rows, u_rows, A * N * 2) ||
                                     overlap(out1_rows, g_rows, A * N * 2));
    if (!u_rows || !large || in_place)
        return launch_grouped_gemm_kn_16(a_rows, w, u_rows, g_rows, out_rows, out1_rows, count, offset, large, A, E, N, K, hidden_act, f16, st);
    const hipError_t e = launch_grouped_gemm_kn_16(a_rows, w, nullptr, nullptr, out_rows, nullptr, count, offset, large, A, E, N, K, hidden_act, f16, st);
    if (e != hipSuccess) return e;
    const unsigned grid = (unsigned)((A * N / 8 + 256 * kRowsPass - 1) / (256 * kRowsPass));
    const auto pass = f16 ? &act_backward_rows_kernel<f16_s> : &act_backward_rows_kernel<bf16_s>;
    pass<<<grid, 256, 0, st>>>((const uint16_t*)u_rows, (const uint16_t*)g_rows, count, offset, E, A, N, hidden_act, (uint16_t*)out_rows, (uint16_t*)out1_rows);
    return hipGetLastError();
}

// out0_rows = a0_rows . w0[e] and out1_rows = a1_rows . w1[e] in one launch, both as launch_expert_gemm_kn gives them.
hipError_t launch_expert_gemm_kn_pair(const void* a0_rows, const void* a1_rows, const void* w0, const void* w1, const int32_t* count,
                                      const int32_t* offset, int64_t A, int E, int N, int K, int dtype, void* out0_rows, void* out1_rows, hipStream_t st) {
    if (dtype == MOE_DTYPE_F32 || !stored_operands_ok(A, N, K)) return hipErrorNotSupported;
    return launch_grouped_gemm_kn_pair_16(a0_rows, a1_rows, w0, w1, out0_rows, out1_rows, count, offset, grouped_kn_large(A, E, N, K, 2), A, E, N, K,
                                          dtype == MOE_DTYPE_FP16, st);
}

static bool wgrad_from_rows(const WgradOperands& w, int64_t A, int dtype, const moe_options& opt) {
    const bool aligned = ((uintptr_t)w.dy | (uintptr_t)w.a | (uintptr_t)w.dw) % 16 == 0;
    return dtype != MOE_DTYPE_F32 && aligned && opt.grouped_tile == MOE_OPT_AUTO && stored_operands_ok(A, w.N, w.K);
}
// dw[e] [N,K] = dy_e^T . a_e, from the rows as they are (product_choice.hpp; not where option grouped_tile asks for a tile) or from
// transposed copies: scratch holds the window offsets and those.
hipError_t launch_expert_wgrad(const void* dy_rows, const void* a_rows, const int32_t* count, const int32_t* offset,
                               int64_t A, int E, int N, int K, int dtype, const moe_options& opt, void* dw, void* scratch,
                               hipStream_t st) {
    const WgradOperands op{dy_rows, a_rows, dw, N, K};
    if (wgrad_from_rows(op, A, dtype, opt)) return launch_wgrad_rows_16(&op, 1, count, offset, wgrad_large(A, E, N, K), E, dtype == MOE_DTYPE_FP16, st);
    const ScratchTables t = scratch_tables(scratch, A, E);
    const int64_t ld = wgrad_ld(A, E);
    const size_t eb = dtype == MOE_DTYPE_F32 ? 4 : 2;
    void* dyT = t.operands;
    void* aT = t.operands + align256((size_t)N * ld * eb);
    backward_tables_kernel<<<1, kMaxExperts, 0, st>>>(count, offset, E, 128, nullptr, nullptr, t.poff);
    const dim3 g1((unsigned)(ld / 64), (unsigned)((N + 63) / 64)), g2((unsigned)(ld / 64), (unsigned)((K + 63) / 64));
    if (dtype == MOE_DTYPE_F32) {
        transpose_rows_padded32_kernel<<<g1, 256, 0, st>>>((const uint32_t*)dy_rows, N, count, offset, t.poff, E, ld, (uint32_t*)dyT);
        transpose_rows_padded32_kernel<<<g2, 256, 0, st>>>((const uint32_t*)a_rows, K, count, offset, t.poff, E, ld, (uint32_t*)aT);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        bool mfma = wgrad_f32_takes_tile(E, N, K);
        if (opt.f32_tile == 0) mfma = false;   // option: keep the vector-ALU kernel
        return (mfma ? launch_wgrad_f32_tile : launch_wgrad_f32)(dyT, aT, dw, t.poff, E, N, K, ld, st);
    }
    transpose_rows_padded_kernel<<<g1, 256, 0, st>>>((const uint16_t*)dy_rows, N, count, offset, t.poff, E, ld, (uint16_t*)dyT);
    transpose_rows_padded_kernel<<<g2, 256, 0, st>>>((const uint16_t*)a_rows, K, count, offset, t.poff, E, ld, (uint16_t*)aT);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return launch_wgrad_16(dyT, aT, dw, t.poff, E, N, K, ld, dtype == MOE_DTYPE_FP16, st);
}

// n weight gradients (1 to 3; of N x K or K x N each) in one launch where all come from the rows as they are, else one after the other.
hipError_t launch_expert_wgrads(const WgradOperands* ops, int n, const int32_t* count, const int32_t* offset, int64_t A, int E, int dtype,
                                const moe_options& opt, void* scratch, hipStream_t st) {
    bool together = true;
    for (int i = 0; i < n; ++i) together = together && wgrad_from_rows(ops[i], A, dtype, opt);
    if (together) return launch_wgrad_rows_16(ops, n, count, offset, wgrad_large(A, E, ops[0].N, ops[0].K, n), E, dtype == MOE_DTYPE_FP16, st);
    for (int i = 0; i < n; ++i) {
        const hipError_t e = launch_expert_wgrad(ops[i].dy, ops[i].a, count, offset, A, E, ops[i].N, ops[i].K, dtype, opt, ops[i].dw, scratch, st);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <class T16, class RAW>
static void launch_act_backward_t(const void* dh, const void* u, const void* g, int64_t n, int act, void* du, void* dg,
                                  hipStream_t st) {
    constexpr int VEC = 16 / (int)sizeof(RAW);
    const uintptr_t bits = (uintptr_t)dh | (uintptr_t)u | (uintptr_t)g | (uintptr_t)du | (uintptr_t)dg;
    if (bits % 16 == 0 && n % VEC == 0) {
        const int grid = (int)std::min<int64_t>((n / VEC + 255) / 256, 65536);
        act_backward_kernel<T16><<<grid, 256, 0, st>>>((const RAW*)dh, (const RAW*)u, (const RAW*)g, (size_t)n, act, (RAW*)du, (RAW*)dg);
    } else {
        const int grid = (int)std::min<int64_t>((n + 255) / 256, 65536);
        act_backward_unaligned_kernel<T16><<<grid, 256, 0, st>>>((const RAW*)dh, (const RAW*)u, (const RAW*)g, (size_t)n, act, (RAW*)du, (RAW*)dg);
    }
}

hipError_t launch_act_backward(const void* dh, const void* u, const void* g, int64_t n, int act, int dtype, void* du,
                               void* dg, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    if (dtype == MOE_DTYPE_F32) launch_act_backward_t<f32_s, float>(dh, u, g, n, act, du, dg, st);
    else if (dtype == MOE_DTYPE_FP16) launch_act_backward_t<f16_s, uint16_t>(dh, u, g, n, act, du, dg, st);
    else launch_act_backward_t<bf16_s, uint16_t>(dh, u, g, n, act, du, dg, st);
    return hipGetLastError();
}

hipError_t launch_bias_grad(const void* dy, const int32_t* count, const int32_t* offset, int E, int N, int dtype, void* db,
                            hipStream_t st) {
    const dim3 grid((unsigned)((N + 255) / 256), (unsigned)E);
    if (dtype == MOE_DTYPE_F32) bias_grad_kernel<f32_s><<<grid, 256, 0, st>>>((const float*)dy, count, offset, N, (float*)db);
    else if (dtype == MOE_DTYPE_FP16) bias_grad_kernel<f16_s><<<grid, 256, 0, st>>>((const uint16_t*)dy, count, offset, N, (uint16_t*)db);
    else bias_grad_kernel<bf16_s><<<grid, 256, 0, st>>>((const uint16_t*)dy, count, offset, N, (uint16_t*)db);
    return hipGetLastError();
}

template <class T16, class RAW>
static void launch_combine_backward_t(const void* dout, const void* y, const int32_t* pair_row, const float* topk_w, int S,
                                      int k, int H, void* dy, float* dw, const RouterGrad& router, hipStream_t st) {
    const uintptr_t bits = (uintptr_t)dout | (uintptr_t)y | (uintptr_t)dy;
    if (bits % 16 == 0)        // (the entry point of the router's share refuses others)
        combine_backward_kernel<T16><<<(S + 3) / 4, 256, 0, st>>>((const RAW*)dout, (const RAW*)y, pair_row, topk_w, S, k, H, (RAW*)dy, dw, router);
    else
        combine_backward_unaligned_kernel<T16><<<S, 256, 0, st>>>((const RAW*)dout, (const RAW*)y, pair_row, topk_w, k, H, (RAW*)dy, dw);
}
static hipError_t combine_backward(const void* dout, const void* y, const int32_t* pair_row, const float* topk_w, int S, int k, int H,
                                   int dtype, void* dy, float* dw, const RouterGrad& router, hipStream_t st) {
    if (S <= 0) return hipSuccess;
    if (dtype == MOE_DTYPE_F32) launch_combine_backward_t<f32_s, float>(dout, y, pair_row, topk_w, S, k, H, dy, dw, router, st);
    else if (dtype == MOE_DTYPE_FP16) launch_combine_backward_t<f16_s, uint16_t>(dout, y, pair_row, topk_w, S, k, H, dy, dw, router, st);
    else launch_combine_backward_t<bf16_s, uint16_t>(dout, y, pair_row, topk_w, S, k, H, dy, dw, router, st);
    return hipGetLastError();
}
hipError_t launch_combine_backward(const void* dout, const void* y, const int32_t* pair_row, const float* topk_w, int S,
                                   int k, int H, int dtype, void* dy, float* dw, hipStream_t st) {
    return combine_backward(dout, y, pair_row, topk_w, S, k, H, dtype, dy, dw, RouterGrad{}, st);
}

// ---- the router's share of a backward pass ----
static int router_ld(int E) { return (E + 15) / 16 * 16; }
size_t router_grad_bytes(int S, int E, int k) { return align256((size_t)S * k * 4) + align256((size_t)S * router_ld(E) * 4) + align256((size_t)S * 4); }
static float* router_dense(void* grad, int S, int k) { return reinterpret_cast<float*>(static_cast<char*>(grad) + align256((size_t)S * k * 4)); }

static int32_t* router_rows(void* grad, int S, int E, int k) {
    return reinterpret_cast<int32_t*>(reinterpret_cast<char*>(router_dense(grad, S, k)) + align256((size_t)S * router_ld(E) * 4));
}

hipError_t launch_combine_backward_router(const void* dout, const void* y, const int32_t* pair_row, const float* topk_w,
                                          const int32_t* topk_idx, const float* logits, int S, int E, int k, int H, int gate_fn, int norm,
                                          int dtype, void* dy, void* grad, hipStream_t st) {
    const RouterGrad r{topk_idx, logits, static_cast<float*>(grad), router_dense(grad, S, k), router_rows(grad, S, E, k), E, router_ld(E), gate_fn, norm};
    return combine_backward(dout, y, pair_row, topk_w, S, k, H, dtype, dy, nullptr, r, st);
}

hipError_t launch_gate_wgrad(const void* x, bool packed, const void* grad, int S, int E, int k, int H, int dtype, void* dgate_w, void* scratch, hipStream_t st) {
    const float* dense = router_dense(const_cast<void*>(grad), S, k);
    const int32_t* row_of = packed ? router_rows(const_cast<void*>(grad), S, E, k) : nullptr;
    // shares: 32 tokens a wavefront, at least enough workgroups for the compute units where there are tokens for them
    const int shares = std::min(std::max((S + 127) / 128, 1), kGateShareMax), n = E * H;
    const dim3 grid((unsigned)((H + 255) / 256), (unsigned)shares, (unsigned)(router_ld(E) / 16));
    float* part = static_cast<float*>(scratch);
    const unsigned sums = (unsigned)((n + 255) / 256);
    if (dtype == MOE_DTYPE_F32) {
        gate_wgrad_kernel<f32_s><<<grid, 256, 0, st>>>((const float*)x, row_of, dense, S, H, E, router_ld(E), part);
        gate_wgrad_sum_kernel<f32_s><<<sums, 256, 0, st>>>(part, shares, n, (float*)dgate_w);
    } else if (dtype == MOE_DTYPE_FP16) {
        gate_wgrad_kernel<f16_s><<<grid, 256, 0, st>>>((const uint16_t*)x, row_of, dense, S, H, E, router_ld(E), part);
        gate_wgrad_sum_kernel<f16_s><<<sums, 256, 0, st>>>(part, shares, n, (uint16_t*)dgate_w);
    } else {
        gate_wgrad_kernel<bf16_s><<<grid, 256, 0, st>>>((const uint16_t*)x, row_of, dense, S, H, E, router_ld(E), part);
        gate_wgrad_sum_kernel<bf16_s><<<sums, 256, 0, st>>>(part, shares, n, (uint16_t*)dgate_w);
    }
    return hipGetLastError();
}

// All operands of the three below are 16-byte aligned (the entry points check it).
hipError_t launch_act_forward(const void* u, const void* g, const int32_t* count, const int32_t* offset, int E, int64_t A, int I,
                              int act, int dtype, void* h, hipStream_t st) {
    const int64_t vecs = A * I / (dtype == MOE_DTYPE_F32 ? 4 : 8);
    if (vecs <= 0) return hipSuccess;
    const int grid = (int)std::min<int64_t>((vecs + 255) / 256, 16384);
    if (dtype == MOE_DTYPE_F32) act_forward_kernel<f32_s><<<grid, 256, 0, st>>>((const float*)u, (const float*)g, count, offset, E, A, I, act, (float*)h);
    else if (dtype == MOE_DTYPE_FP16) act_forward_kernel<f16_s><<<grid, 256, 0, st>>>((const uint16_t*)u, (const uint16_t*)g, count, offset, E, A, I, act, (uint16_t*)h);
    else act_forward_kernel<bf16_s><<<grid, 256, 0, st>>>((const uint16_t*)u, (const uint16_t*)g, count, offset, E, A, I, act, (uint16_t*)h);
    return hipGetLastError();
}

hipError_t launch_dispatch_rows(const void* x, const int32_t* token_indices, int64_t A, int S, int H, int dtype, void* rows,
                                hipStream_t st) {
    if (A <= 0) return hipSuccess;
    const int row_vec = H * (dtype == MOE_DTYPE_F32 ? 4 : 2) / 16;
    dispatch_rows_kernel<<<(unsigned)((A + 3) / 4), 256, 0, st>>>((const uint4*)x, token_indices, A, row_vec, S, (uint4*)rows);
    return hipGetLastError();
}

// topk_idx, grad, gate_w: null, or what adds the router's share to the tokens' gradient.
hipError_t launch_dispatch_backward(const void* a, const void* b, const int32_t* pair_row, int S, int k, int H, int dtype,
                                    void* dx, const int32_t* topk_idx, const void* grad, const void* gate_w, hipStream_t st) {
    if (S <= 0) return hipSuccess;
    const int piece = 64 * 16 / (dtype == MOE_DTYPE_F32 ? 4 : 2), pieces = (H + piece - 1) / piece;
    const int64_t blocks = ((int64_t)S * pieces + 3) / 4;
    if (blocks > INT32_MAX) return hipErrorInvalidValue;
    const unsigned grid = (unsigned)blocks;
    const float* dl = static_cast<const float*>(grad);
    if (dtype == MOE_DTYPE_F32) dispatch_backward_kernel<f32_s><<<grid, 256, 0, st>>>((const float*)a, (const float*)b, pair_row, S, k, H, pieces, (float*)dx, topk_idx, dl, (const float*)gate_w);
    else if (dtype == MOE_DTYPE_FP16) dispatch_backward_kernel<f16_s><<<grid, 256, 0, st>>>((const uint16_t*)a, (const uint16_t*)b, pair_row, S, k, H, pieces, (uint16_t*)dx, topk_idx, dl, (const uint16_t*)gate_w);
    else dispatch_backward_kernel<bf16_s><<<grid, 256, 0, st>>>((const uint16_t*)a, (const uint16_t*)b, pair_row, S, k, H, pieces, (uint16_t*)dx, topk_idx, dl, (const uint16_t*)gate_w);
    return hipGetLastError();
}

}  // namespace moe355
