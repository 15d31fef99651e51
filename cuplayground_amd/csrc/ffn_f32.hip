// Expert FFN in fp32 (torch_dtype 0): the reference's tile GEMM contract, C = act(A.B^T + bias)
// (mma.cuh:46-179; its only instantiated case is fp32 + ReLU, mma.cuh:378-384).
// The kernels of small and ragged fp32 layers (large ones take ffn_f32_tile.hip): a plain LDS-tiled FMA kernel, 64x64 output
// tile, 16-wide K slabs, 256 threads with a 4x4 register block each, and for layers of few rows or few tasks wavefronts that
// stream weights into the fp32 matrix instructions.  Task decoding, dispatch-by-gather and the
// phase dependency protocol are shared with the bf16 path.
#include "ffn_common.hpp"

namespace moe355 {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int FBM = 64, FBN = 64, FBK = 16, FPAD = 4;

struct TaskPtrsF {
    const float* a_base;
    const int32_t* gather;
    int64_t a_row0;
    int a_ld;
    int b_ld;          // row pitch of b0 / b1 (K, except for windows of a wider matrix)
    const float* b0;
    const float* b1;
    const float* bias0;
    const float* bias1;
    float* c_base;
    int N, K, rows, n0, act;
    bool swiglu;
    bool publish;   // rows are read by other workgroups of the same launch
};

__device__ __forceinline__ void gemm_tile_f32(const TaskPtrsF& p, float (*As)[FBM + FPAD], float (*Bs)[FBN + FPAD]) {
    const int tid = threadIdx.x;
    const int ty = tid >> 4, tx = tid & 15;
    const int lrow = tid >> 2, lk = (tid & 3) * 4;

    int ar = lrow < p.rows ? lrow : 0;
    const int64_t src_row = p.gather ? (int64_t)p.gather[ar] : p.a_row0 + ar;
    const float* a_src = p.a_base + src_row * p.a_ld + lk;

    int col;
    const float* bbase = p.b0;
    if (p.swiglu) {
        col = p.n0 + (lrow & 31);
        bbase = (lrow >> 5) ? p.b0 : p.b1;      // tile rows 0..31 gate, 32..63 up
    } else {
        col = p.n0 + lrow;
    }
    if (col >= p.N) col = p.N - 1;
    const float* b_src = bbase + (int64_t)col * p.b_ld + lk;

    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[i][q] = 0.0f;

    for (int k0 = 0; k0 < p.K; k0 += FBK) {
        const float4 av = *reinterpret_cast<const float4*>(a_src + k0);
        const float4 bv = *reinterpret_cast<const float4*>(b_src + k0);
        __syncthreads();
        As[lk + 0][lrow] = av.x; As[lk + 1][lrow] = av.y; As[lk + 2][lrow] = av.z; As[lk + 3][lrow] = av.w;
        Bs[lk + 0][lrow] = bv.x; Bs[lk + 1][lrow] = bv.y; Bs[lk + 2][lrow] = bv.z; Bs[lk + 3][lrow] = bv.w;
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < FBK; ++kk) {
            const float4 a4 = *reinterpret_cast<const float4*>(&As[kk][ty * 4]);
            const float2 b01 = *reinterpret_cast<const float2*>(&Bs[kk][tx * 2]);
            const float2 b23 = *reinterpret_cast<const float2*>(&Bs[kk][32 + tx * 2]);
            const float a[4] = {a4.x, a4.y, a4.z, a4.w};
            const float b[4] = {b01.x, b01.y, b23.x, b23.y};
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q) acc[i][q] = __builtin_fmaf(a[i], b[q], acc[i][q]);
        }
    }

#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = ty * 4 + i;
        if (m >= p.rows) continue;
        float* crow = p.c_base + (int64_t)m * p.N;
        if (p.swiglu) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int c = p.n0 + tx * 2 + q;
                if (c >= p.N) continue;
                float g = acc[i][q], u = acc[i][q + 2];
                if (p.bias1) g = g + p.bias1[c];
                if (p.bias0) u = u + p.bias0[c];
                const float v = silu(g) * u;
                if (p.publish) publish4(crow + c, __float_as_uint(v)); else crow[c] = v;
            }
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int c = p.n0 + (q >> 1) * 32 + tx * 2 + (q & 1);
                if (c >= p.N) continue;
                float u = acc[i][q];
                if (p.bias0) u = u + p.bias0[c];
                const float v = act_apply(u, p.act);
                if (p.publish) publish4(crow + c, __float_as_uint(v)); else crow[c] = v;
            }
        }
    }
}

// ---- the weight streamer ----
// 64 rows x 64 columns of one projection (SwiGLU: of both, 64 gate and 64 up rows) on v_mfma_f32_16x16x4_f32 without LDS or
// barriers.  A wavefront owns 16 columns over the whole contraction dimension: weight rows as the "A" operand, up to NT
// groups of 16 token rows as "B", each fetched as 16 bytes a lane and 16 values of k an instruction, the next chunk of
// weights in flight while this one is multiplied.  Lane group g holds k = 4 g .. 4 g + 3 of a slab, and matrix instruction j
// multiplies element j of every lane group: a permutation of the slab's k that both operands share.  Two accumulators per
// output element (even and odd slabs), added at the end.
//
// What bounds a small layer is latency: 128 rows on 8 experts of 256 x 512 are 1 us of arithmetic for 64 and 32 tasks.  The
// LDS-tiled FMA kernel above waits for memory and two barriers every 16 values of k and always computes 64 rows;
// here 8 KB of weights a wavefront are in flight (eight slabs of one matrix, four of SwiGLU's two; half of that for blocks of more than
// 32 rows, whose token rows take the registers), nothing is waited for but the operands, and groups of 16 rows that a block does not have cost nothing.  Whole layer, that kernel -> this one, us: 128 tokens, 8 experts of 256 x 512, GELU 67.6 ->
// 33.2; 40 tokens top-2 of 16, 128 x 768 76 -> 34; 192 tokens, 4 of 448 x 640 90 -> 72; 537 tokens, 8 of 384 x 256 64 -> 52; 332
// tokens, one of 1024 x 4096 331 -> 255; 16 tokens, 8 of 4096 x 14336, SwiGLU 2990 -> 1020.  Error against float64: 5.2e-7 -> 3.7e-7
// (first), 1.0e-6 -> 7.0e-7 (fifth).  Where full blocks keep the chip busy it loses to the LDS kernel, which reads a token row
// once for 64 columns and not for 16 (api.hip: ffn_plan has the line).
template <int MATS, int NT>
__device__ __forceinline__ void stream_tile_f32(const TaskPtrsF& p) {
    constexpr int U = (NT >= 4 ? 4 : 8) / MATS;      // slabs of 16 in flight
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int idx = lane & 15, kg = lane >> 4;
    const int c0 = p.n0 + 16 * wave;                 // N is a multiple of 64: a wavefront's columns exist together or not at all
    if (c0 >= p.N) return;

    const float* wp[MATS];
#pragma unroll
    for (int m = 0; m < MATS; ++m) wp[m] = (m ? p.b1 : p.b0) + (int64_t)(c0 + idx) * p.b_ld + 4 * kg;
    // rows behind the block's last one read row 0 again and are never stored
    const float* xp[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const int r = 16 * i + idx < p.rows ? 16 * i + idx : 0;
        xp[i] = p.a_base + (p.gather ? (int64_t)p.gather[r] : p.a_row0 + r) * p.a_ld + 4 * kg;
    }

    f32x4 acc[2][MATS][NT];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int m = 0; m < MATS; ++m)
#pragma unroll
            for (int i = 0; i < NT; ++i) acc[h][m][i] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int slabs = p.K >> 4, full = slabs / U, left = slabs - full * U;
    f32x4 w[MATS][U], wn[MATS][U], x[NT][U];
    // slabs behind the last one read it again (and are not multiplied)
    auto load_w = [&](f32x4 (&d)[MATS][U], int s0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = min(s0 + u, slabs - 1) << 4;
#pragma unroll
            for (int m = 0; m < MATS; ++m) d[m][u] = *reinterpret_cast<const f32x4*>(wp[m] + k);
        }
    };
    auto load_x = [&](int s0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = min(s0 + u, slabs - 1) << 4;
#pragma unroll
            for (int i = 0; i < NT; ++i) x[i][u] = *reinterpret_cast<const f32x4*>(xp[i] + k);
        }
    };
    auto multiply = [&](int u) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int m = 0; m < MATS; ++m)
#pragma unroll
                for (int i = 0; i < NT; ++i)
                    acc[u & 1][m][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[m][u][j], x[i][u][j], acc[u & 1][m][i], 0, 0, 0);
    };
    load_w(w, 0);
    for (int c = 0; c < full; ++c) {
        load_x(c * U);                               // first: loads return in order, and these are needed first
        if ((c + 1) * U < slabs) load_w(wn, (c + 1) * U);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; ++u) multiply(u);
#pragma unroll
        for (int m = 0; m < MATS; ++m)
#pragma unroll
            for (int u = 0; u < U; ++u) w[m][u] = wn[m][u];
    }
    if (left) {
        load_x(full * U);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (u < left) multiply(u);
    }

    // this lane holds token rows 16 i + idx, columns c0 + 4 kg ..+3
    const int col = c0 + 4 * kg;
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const int row = 16 * i + idx;
        if (row >= p.rows) continue;
        float v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float u = acc[0][0][i][q] + acc[1][0][i][q];
            if (p.bias0) u = u + p.bias0[col + q];
            if constexpr (MATS == 2) {
                float g = acc[0][1][i][q] + acc[1][1][i][q];
                if (p.bias1) g = g + p.bias1[col + q];
                v[q] = silu(g) * u;
            } else {
                v[q] = act_apply(u, p.act);
            }
        }
        float* out = p.c_base + (int64_t)row * p.N + col;
        if (p.publish) {
            publish8(out, __float_as_uint(v[0]), __float_as_uint(v[1]));
            publish8(out + 2, __float_as_uint(v[2]), __float_as_uint(v[3]));
        } else {
            *reinterpret_cast<f32x4*>(out) = f32x4{v[0], v[1], v[2], v[3]};
        }
    }
}

// Groups of 16 rows that the block does not have are neither read nor multiplied.
__device__ __forceinline__ void stream_rows_f32(const TaskPtrsF& p) {
    if (p.swiglu) {
        if (p.rows <= 16) stream_tile_f32<2, 1>(p);
        else if (p.rows <= 32) stream_tile_f32<2, 2>(p);
        else stream_tile_f32<2, 4>(p);
    } else {
        if (p.rows <= 16) stream_tile_f32<1, 1>(p);
        else if (p.rows <= 32) stream_tile_f32<1, 2>(p);
        else stream_tile_f32<1, 4>(p);
    }
}

template <bool STREAM>
__device__ __forceinline__ TaskPtrsF resolve_f32(const FfnArgs& a, const Task& t, bool publish) {
    TaskPtrsF p;
    const int64_t HI = (int64_t)a.H * a.I;
    const bool sw = a.act == MOE_ACT_SWIGLU;
    if (t.phase == 0) {
        p.a_base = (const float*)a.x;
        p.gather = a.token_indices + t.row0;
        p.a_row0 = 0;
        p.a_ld = a.H;
        p.b_ld = a.H;
        p.b0 = (const float*)a.w_up + t.expert * HI;
        p.b1 = sw ? (const float*)a.w_gate + t.expert * HI : nullptr;
        p.bias0 = a.b_up ? (const float*)a.b_up + (int64_t)t.expert * a.I : nullptr;
        p.bias1 = (sw && a.b_gate) ? (const float*)a.b_gate + (int64_t)t.expert * a.I : nullptr;
        p.c_base = (float*)a.h + (int64_t)t.row0 * a.I;
        p.N = a.I;
        p.K = a.H;
        p.n0 = t.ntile * (sw && !STREAM ? FBN / 2 : FBN);
        p.act = a.act;
        p.swiglu = sw;
        p.publish = publish;
    } else {
        p.a_base = (const float*)a.h;
        p.gather = nullptr;
        p.a_row0 = t.row0;
        p.a_ld = a.I;
        p.b_ld = a.I;
        p.b0 = (const float*)a.w_down + t.expert * HI;
        p.b1 = nullptr;
        p.bias0 = a.b_down ? (const float*)a.b_down + (int64_t)t.expert * a.H : nullptr;
        p.bias1 = nullptr;
        p.c_base = (float*)a.y + (int64_t)t.row0 * a.H;
        p.N = a.H;
        p.K = a.I;
        p.n0 = t.ntile * FBN;
        p.act = MOE_ACT_NONE;
        p.swiglu = false;
        p.publish = publish;
    }
    p.rows = t.rows;
    return p;
}

template <bool STREAM>
__global__ __launch_bounds__(256, STREAM ? 3 : 1) void ffn_tiled_f32_kernel(FfnArgs a, int phase) {
    __shared__ __align__(16) float As[STREAM ? 1 : FBK][FBM + FPAD];
    __shared__ __align__(16) float Bs[STREAM ? 1 : FBK][FBN + FPAD];
    Task t;
    __shared__ int s_list[1 + FBM];
    if (phase == 0) zero_unrouted_rows(a, 4);
    if (!tiled_task(a, phase, blockIdx.x, t)) return;
    const TaskPtrsF p = resolve_f32<STREAM>(a, t, phase == 1 && a.arrive);
    if constexpr (STREAM) stream_rows_f32(p);
    else gemm_tile_f32(p, As, Bs);
    if (phase == 1 && a.arrive) combine_arrivals<float>(combine_args(a), t.row0, t.rows, t.ntile, p.n0, FBN, s_list);
}

template <bool STREAM>
__global__ __launch_bounds__(256, STREAM ? 3 : 1) void ffn_persistent_f32_kernel(FfnArgs a) {
    __shared__ __align__(16) float As[STREAM ? 1 : FBK][FBM + FPAD];
    __shared__ __align__(16) float Bs[STREAM ? 1 : FBK][FBN + FPAD];
    __shared__ int s_task, s_ok;
    __shared__ int s_cmb[kCombineLds];
    __shared__ int s_list[1 + FBM];
    queue_kernel_entry();
    queue_clock_stamp(a.wg_clock, 0);
    zero_unrouted_rows(a, 4);
    const int ids = a.q->ids_queue;
    const int nseg = a.q->nseg;
    const int nnt0 = a.seg_phase0[0].nnt;
    QueueCursor cur = queue_cursor(a.groups);
    Task t;
    while (next_task(a, cur, &s_task, ids, nseg, nnt0, t)) {
        int ok = 1;
        if (t.phase == 1) ok = wait_phase0_done(a.done0, t.mtile, nnt0, a.spin_limit, a.q, a.host_stall, &s_ok);
        const TaskPtrsF p = resolve_f32<STREAM>(a, t, t.phase == 0 || publish_y(a));
        const long long started = trace_clock(a.task_trace);
        if (ok) {
            if constexpr (STREAM) stream_rows_f32(p);
            else gemm_tile_f32(p, As, Bs);
        } else poison_tile(p.c_base, p.rows, p.N, p.n0, FBN, 4);
        if (a.task_trace) trace_task(a.task_trace, a.task_trace_cap, t.phase, t.expert, t.mtile, t.ntile, t.rows, started);
        if (t.phase == 0) signal_phase0_done(a.done0, t.mtile);
        else after_down_tile<float>(a, t.row0, t.rows, t.mtile, t.ntile, p.n0, FBN, s_list);
    }
    if (a.combined) combine_while_idle_narrow<float>(sweep_args(a), &s_task, s_cmb);
    queue_clock_stamp(a.wg_clock, 1);
}

__global__ __launch_bounds__(256) void gemm_dense_f32_kernel(const float* A, const float* B, const float* bias,
                                                             float* C, int M, int N, int K, int act) {
    __shared__ __align__(16) float As[FBK][FBM + FPAD];
    __shared__ __align__(16) float Bs[FBK][FBN + FPAD];
    TaskPtrsF p;
    const int row0 = blockIdx.y * FBM;
    p.a_base = A; p.gather = nullptr; p.a_row0 = row0; p.a_ld = K; p.b_ld = K;
    p.b0 = B; p.b1 = nullptr; p.bias0 = bias; p.bias1 = nullptr;
    p.c_base = C + (int64_t)row0 * N;
    p.N = N; p.K = K; p.rows = min(FBM, M - row0); p.n0 = blockIdx.x * FBN; p.act = act; p.swiglu = false; p.publish = false;
    gemm_tile_f32(p, As, Bs);
}

// Grouped product over packed expert-major rows (backward.hip): out[r,:] = act(a_rows[r,:] . w[e(r)]^T + bias[e(r)]),
// one workgroup per (row block of 64 from `mtiles`, 64 output columns).
__global__ __launch_bounds__(256) void grouped_gemm_f32_kernel(const float* a_rows, const float* w, const float* bias,
                                                               float* out, const MTile* mtiles, const int32_t* num_mtiles,
                                                               int nnt, int N, int K, int act) {
    __shared__ __align__(16) float As[FBK][FBM + FPAD];
    __shared__ __align__(16) float Bs[FBK][FBN + FPAD];
    const int mt = blockIdx.x / nnt, nt = blockIdx.x % nnt;
    if (mt >= *num_mtiles) return;
    const MTile m = mtiles[mt];
    TaskPtrsF p;
    p.a_base = a_rows; p.gather = nullptr; p.a_row0 = m.row0; p.a_ld = K; p.b_ld = K;
    p.b0 = w + (int64_t)m.expert * N * K; p.b1 = nullptr;
    p.bias0 = bias ? bias + (int64_t)m.expert * N : nullptr; p.bias1 = nullptr;
    p.c_base = out + (int64_t)m.row0 * N;
    p.N = N; p.K = K; p.rows = m.rows; p.n0 = nt * FBN; p.act = act; p.swiglu = false; p.publish = false;
    gemm_tile_f32(p, As, Bs);
}

// Weight gradient of one expert: dw[e] [N,K] = dyT[:, window e] . aT[:, window e]^T, the windows being the expert's
// packed rows as columns of the transposed operands (zero padded to a multiple of 128, pitch ld).
// grid = (ceil(K / 64), ceil(N / 64), E).
__global__ __launch_bounds__(256) void wgrad_f32_kernel(const float* dyT, const float* aT, float* dw, const int32_t* poff,
                                                        int N, int K, int64_t ld) {
    __shared__ __align__(16) float As[FBK][FBM + FPAD];
    __shared__ __align__(16) float Bs[FBK][FBN + FPAD];
    const int e = blockIdx.z, row0 = blockIdx.y * FBM;
    TaskPtrsF p;
    p.a_base = dyT + poff[e]; p.gather = nullptr; p.a_row0 = row0; p.a_ld = (int)ld; p.b_ld = (int)ld;
    p.b0 = aT + poff[e]; p.b1 = nullptr; p.bias0 = nullptr; p.bias1 = nullptr;
    p.c_base = dw + (int64_t)e * N * K + (int64_t)row0 * K;
    p.N = K; p.K = poff[e + 1] - poff[e]; p.rows = min(FBM, N - row0); p.n0 = blockIdx.x * FBN; p.act = MOE_ACT_NONE;
    p.swiglu = false; p.publish = false;
    gemm_tile_f32(p, As, Bs);
}

}  // namespace

int f32_block_m() { return FBM; }
int f32_block_n() { return FBN; }

template <bool STREAM>
static void launch_tiled(const FfnArgs& a, int max_mtiles, int nnt0, int nnt1, hipStream_t st) {
    ffn_tiled_f32_kernel<STREAM><<<tiled_grid(max_mtiles, nnt0, a.groups), 256, 0, st>>>(a, 0);
    ffn_tiled_f32_kernel<STREAM><<<tiled_grid(max_mtiles, nnt1, a.groups), 256, 0, st>>>(a, 1);
}
hipError_t launch_ffn_tiled_f32(const FfnArgs& a, bool stream, int max_mtiles, int nnt0, int nnt1, hipStream_t st) {
    if (stream) launch_tiled<true>(a, max_mtiles, nnt0, nnt1, st);
    else launch_tiled<false>(a, max_mtiles, nnt0, nnt1, st);
    return hipGetLastError();
}

hipError_t launch_ffn_persistent_f32(const FfnArgs& a, bool stream, int blocks, hipStream_t st) {
    if (stream) ffn_persistent_f32_kernel<true><<<blocks, 256, 0, st>>>(a);
    else ffn_persistent_f32_kernel<false><<<blocks, 256, 0, st>>>(a);
    return hipGetLastError();
}

hipError_t launch_gemm_dense_f32(const void* A, const void* B, const void* bias, void* C, int64_t M, int64_t N,
                                 int64_t K, int act, hipStream_t st) {
    const dim3 grid((unsigned)((N + FBN - 1) / FBN), (unsigned)((M + FBM - 1) / FBM));
    gemm_dense_f32_kernel<<<grid, 256, 0, st>>>((const float*)A, (const float*)B, (const float*)bias, (float*)C,
                                                (int)M, (int)N, (int)K, act);
    return hipGetLastError();
}

hipError_t launch_grouped_gemm_f32(const void* a_rows, const void* w, const void* bias, void* out, const MTile* mtiles,
                                   const int32_t* num_mtiles, int max_mtiles, int N, int K, int act, hipStream_t st) {
    const int nnt = (N + FBN - 1) / FBN;
    grouped_gemm_f32_kernel<<<(unsigned)max_mtiles * nnt, 256, 0, st>>>((const float*)a_rows, (const float*)w,
                                                                        (const float*)bias, (float*)out, mtiles,
                                                                        num_mtiles, nnt, N, K, act);
    return hipGetLastError();
}

hipError_t launch_wgrad_f32(const void* dyT, const void* aT, void* dw, const int32_t* poff, int E, int N, int K, int64_t ld,
                            hipStream_t st) {
    const dim3 grid((unsigned)((K + FBN - 1) / FBN), (unsigned)((N + FBM - 1) / FBM), (unsigned)E);
    wgrad_f32_kernel<<<grid, 256, 0, st>>>((const float*)dyT, (const float*)aT, (float*)dw, poff, N, K, ld);
    return hipGetLastError();
}

}  // namespace moe355
