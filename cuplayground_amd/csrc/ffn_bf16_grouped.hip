// Products on the 16-bit tiles (ffn_bf16_tile.hpp): dense operands, packed rows by expert (a layer's two launches too), weight gradients.
#include <algorithm>

#include "ffn_bf16_tile.hpp"
#include "grouped_task.hpp"

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
// (the smaller tile takes two thirds of the larger one's time at 16 slabs, three quarters at 32: tile_task_us; the other half of the
// larger one would multiply zeros).
// KN: the weights are stored with k as their slow index.
template <bool F16_, int BIG_, bool KN_ = false>
struct RowSplit {
    static constexpr bool F16 = F16_, HAND = true, KN = KN_;
    static constexpr int BIG = BIG_, BN = 256, THREADS = 256;
    using TH = Tile<128, 256, 1, 4, 2, F16_, false, KN_>;
    using TB = typename std::conditional<BIG_ == 256, Tile<256, 256, 2, 2, 2, F16_, false, KN_>, TH>::type;
    static constexpr int LDS_BYTES = TB::LDS_BYTES;
    static_assert(TH::LDS_BYTES <= LDS_BYTES, "one dynamic LDS block for both");
};
// The 128 x 128 tile of the general loop.
template <bool F16_>
struct PlainSplit {
    static constexpr bool F16 = F16_, HAND = false, KN = false;
    using TB = Tile<128, 128, 2, 2, 2, F16_>;
    static constexpr int BIG = 128, BN = 128, THREADS = 256, LDS_BYTES = TB::LDS_BYTES;
};

// What a grouped product does with its sums: one kernel each, so that a tile's code is a slab loop and one epilogue (with three of
// them a kernel of several tiles is twice the instruction cache).
enum : int { kSums = 0, kGelu = 2, kSwiglu = 3, kDeriv = 4 };      // sums or ReLU; GELU; SwiGLU; the activation's derivative
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

// Grouped GEMM on packed expert-major rows: out[r,:] = act(a[r,:] . w[e(r)]^T + bias[e(r)]) -- the
// reference's tile GEMM (mma.cuh:46-179) once per expert.  With the weight handed over in its K-major view this is the data
// gradient of a projection (dX = dY . W).  DERIV: that of the down projection with the activation's derivative in its epilogue,
// which hands on dU (and dG) instead of dH.  With gather and w1 the up projection of a layer.  One workgroup per tile (grouped_task).
// Two products of one shape (a training step's up and gate projections, and their data gradients) share a launch as one of twice the
// columns, the second product's behind the first's: each would end in a round of few tasks.  Two launches / one, us, projections and
// data gradients: 16 experts of 2048 x 1408, 750 rows each 191 / 156 and 161 / 143; 4 of 2048 x 2560, 4096 rows 297 / 268, 283 / 269; 8 of
// 1280 x 1664, 256 rows 42 / 33, 48 / 26; 16 of 1152 x 1920, 175 rows 46 / 36, 53 / 44; 16 of 1024 x 2560, 62 rows 39 / 40, 62 / 34.
struct GroupedArgs {
    const uint16_t* a_rows;      // packed rows, or with gather the tokens
    const uint16_t* w;           // [E, N, K] (KN: [E, K, N])
    const uint16_t* bias;        // or null
    const uint16_t* u_rows;      // DERIV: the saved projections ...
    const uint16_t* g_rows;      // ... and, with SwiGLU, the gate's
    uint16_t* out;               // rows of the result (DERIV: dU)
    uint16_t* out1;              // DERIV, SwiGLU: dG
    const int32_t* count;
    const int32_t* offset;
    int E, N, K, act;            // act: the epilogue's activation (DERIV: the layer's hidden_act)
    uint32_t a_bytes;
    // a layer's up projection:
    const int32_t* gather;       // null, or the token of every packed row
    const uint16_t* w1;          // SwiGLU: the gate's weights ...
    const uint16_t* bias1;       // ... and biases, or null
    const uint16_t* a1_rows;     // kSums with out1: a second product of the same shape, a1_rows and w1 into out1
};
template <class P, int EPI>
__global__ __launch_bounds__(P::THREADS) void grouped_gemm_kernel(GroupedArgs a) {
    constexpr bool DERIV = EPI == kDeriv, SWIGLU = EPI == kSwiglu;
    constexpr int COLS = SWIGLU ? P::BN / 2 : P::BN;      // half of a SwiGLU tile's weight rows are gate rows
    extern __shared__ __align__(16) unsigned char smem[];
    const int N = a.N, K = a.K;
    const int cols = (N + COLS - 1) / COLS;
    const bool two = EPI == kSums && a.out1;
    GroupedTask t;
    if (!grouped_task<P::BIG>(a.count, a.offset, a.E, two ? 2 * cols : cols, blockIdx.x, t)) return;
    const bool second = two && t.ctile >= cols;
    if (second) t.ctile -= cols;
    const int64_t at = (int64_t)t.row0 * N;
    TaskPtrs p;
    p.a_base = second ? a.a1_rows : a.a_rows;
    p.gather = a.gather ? a.gather + t.row0 : nullptr;
    p.a_row0 = a.gather ? 0 : t.row0;
    p.a_ld = K;
    p.b0 = (second ? a.w1 : a.w) + (int64_t)t.expert * N * K;
    p.b1 = SWIGLU ? a.w1 + (int64_t)t.expert * N * K : nullptr;
    p.b_ld = K;
    p.bias0 = !DERIV && a.bias ? a.bias + (int64_t)t.expert * N : nullptr;
    p.bias1 = SWIGLU && a.bias1 ? a.bias1 + (int64_t)t.expert * N : nullptr;
    p.c_base = (second ? a.out1 : a.out) + at;
    p.N = N;
    p.K = K;
    p.rows = t.rows;
    p.n0 = t.ctile * COLS;
    p.act = DERIV ? MOE_ACT_NONE : a.act;
    p.swiglu = SWIGLU;
    p.publish = false;
    p.a_extent = a.a_bytes;
    p.b_extent = (uint32_t)((int64_t)N * K * 2);
    if constexpr (P::KN) {
        p.b0 += p.n0;
        p.b_ld = N;
        p.b_extent -= (uint32_t)p.n0 * 2;
    }
    p.part = nullptr; p.part_cnt = nullptr; p.kparts = 1; p.kpart = 0; p.poison = false;
    p.deriv = DERIV ? 1 + a.act : 0;
    p.aux0 = DERIV ? a.u_rows + at : nullptr;
    p.aux1 = DERIV && a.g_rows ? a.g_rows + at : nullptr;
    p.c1_base = DERIV && a.out1 ? a.out1 + at : nullptr;
    grouped_tile<P, EPI>(p, smem);
}

// ---- weight gradients from the packed rows as they lie ----
//
// C[i, j] = sum over k of A(i, k) B(j, k) on 128 x 128 tiles, both operands stored with k as the slow index (dW[e] = dY_e^T . X_e).
// An operand is turned round on its way through the registers: a thread fetches 16 bytes of four consecutive k and writes, for each
// of the eight i, the four values of k side by side (one byte permute a dword), so that LDS holds what it holds for the other
// tiles and nothing else is ever written to memory.
template <bool F16_>
struct ProdTile {
    static constexpr int BM = 128, BN = 128, WM = 2, WN = 2, NS = 2, THREADS = 256, TM = 4, TN = 4, WB = 64;
    static constexpr bool F16 = F16_, RING = false, HALF = false, HAND = true, TRA = false;
    static constexpr int STAGE_BYTES = (BM + BN) * kRowBytes;
    static constexpr int STAGING_BYTES = 4 * 16 * (TN * 32 + 16);
    static constexpr int LDS_BYTES = NS * STAGE_BYTES + STAGING_BYTES;
    static_assert(2 * LDS_BYTES <= 160 * 1024, "two workgroups per compute unit");
};
// An operand of one tile: 128 rows i (or columns j) from `base` on.
struct ProdOperand {
    const uint16_t* base;
    int ld;                // elements between consecutive k
    uint32_t extent;       // bytes from base that exist; loads behind read zeros
};
// LDS: 128-byte rows of 64 k, 16-byte piece c of row i at c ^ prod_swizzle(i).  The 16 rows of a fragment read meet all banks, and
// so do eight rows that lie eight apart, which is what a transposed operand writes at a time.
__device__ __forceinline__ int prod_swizzle(int i) { return ((i >> 1) ^ (i >> 4)) & 7; }
struct ProdLoads {
    uint32_t off[4];       // rows behind the operand's last one lie behind its extent, whatever the tile
    int put;
    __device__ __forceinline__ ProdLoads(int ld, int tid) {
        // Eight lanes in a row fetch 128 bytes in a row: the address unit takes four neighbouring lanes a cycle only where
        // their addresses follow each other, else one (with the lanes of a row eight apart: 64 cycles a request, the unit busy
        // 94 % of the time, 1.6 times the kernel's time).
        const int lane = tid & 63, wave = tid >> 6;
        const int kq = (lane >> 3) + 8 * (wave & 1), ig = (lane & 7) + 8 * (wave >> 1);
#pragma unroll
        for (int q = 0; q < 4; ++q) off[q] = (uint32_t)((4 * kq + q) * ld + 8 * ig) * 2;
        put = ig * 8 * kRowBytes + (((kq >> 1) ^ prod_swizzle(8 * ig)) << 4) + (kq & 1) * 8;
    }
    // slab s of 64 k; k behind the extent are zeros.
    __device__ __forceinline__ void load(const ProdOperand& o, int slab, u32x4 (&d)[4]) const {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(o.base), 0, (int)o.extent, 0x00020000);
        const uint32_t k = (uint32_t)(slab * kBK) * o.ld * 2;
#pragma unroll
        for (int q = 0; q < 4; ++q) d[q] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(off[q] + k), 0, 0));
    }
    __device__ __forceinline__ void store(const u32x4 (&d)[4], unsigned char* st) const {
#pragma unroll
        for (int j = 0; j < 8; ++j) {      // row i = 8 ig + j: its swizzle differs from that of 8 ig by j >> 1
            const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
            const u32x2 v = {__builtin_amdgcn_perm(d[1][j >> 1], d[0][j >> 1], sel), __builtin_amdgcn_perm(d[3][j >> 1], d[2][j >> 1], sel)};
            *reinterpret_cast<u32x2*>(st + ((put ^ ((j >> 1) << 4)) + j * kRowBytes)) = v;
        }
    }
};

// The same in every lane, and said so: else each load loops over the lanes.
__device__ __forceinline__ ProdOperand prod_uniform(const ProdOperand& o) {
    const uint64_t v = (uint64_t)o.base;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v), hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return ProdOperand{(const uint16_t*)(((uint64_t)hi << 32) | lo), __builtin_amdgcn_readfirstlane(o.ld), (uint32_t)__builtin_amdgcn_readfirstlane((int)o.extent)};
}

// One tile of a launch: its operands and how many slabs of 64 k it has (at least one).
struct ProdJob {
    ProdOperand a, b;
    int slabs;
};

// The slab loop of one tile.  What bounds it: LDS (a 64 x 64 wavefront tile reads 16 KB of fragments a slab at 256 bytes a cycle,
// the slab's 32 KB are written at 128), the address unit (64 bytes a cycle) and the matrix instructions, each about half of the
// time; two workgroups share a compute unit and fill each other's waits.  0.85 PFLOP/s with 4096 rows an expert (a weight
// gradient of 4 x 2048 x 2560), 0.65 with 512 (of 16 x 2048 x 2048).  (Workgroups that stay and
// request the next tile's first slabs under this one's last: no faster, what they save at the ends of tiles they lose in the
// last round of an uneven number of tiles.)
template <class T>
__device__ __forceinline__ void prod_slabs(const ProdJob& job, unsigned char* smem, f32x4 (&acc)[T::TM][T::TN]) {
    constexpr int D = 2;                       // slabs on their way in registers
    typedef typename std::conditional<T::F16, f16x8, bf16x8>::type frag_t;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / T::WN, wn = wave % T::WN;
    const ProdLoads la(job.a.ld, tid);
    const ProdLoads lb(job.b.ld, tid);
    const int slabs = job.slabs;
    const int frow = lane & 15, fk = lane >> 4, sw = (frow >> 1) & 7;
    int get_a[T::TM], get_b[T::TN];            // this lane's pieces of k half 0; those of half 1 lie 64 bytes up or down
#pragma unroll
    for (int i = 0; i < T::TM; ++i) get_a[i] = (16 * (wm * T::TM + i) + frow) * kRowBytes + ((fk ^ sw ^ ((wm * T::TM + i) & 7)) << 4);
#pragma unroll
    for (int j = 0; j < T::TN; ++j) get_b[j] = (T::BM + 16 * (wn * T::TN + j) + frow) * kRowBytes + ((fk ^ sw ^ ((wn * T::TN + j) & 7)) << 4);
#pragma unroll
    for (int i = 0; i < T::TM; ++i)
#pragma unroll
        for (int j = 0; j < T::TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 ra[D][4], rb[D][4];
    frag_t fa[2][T::TM], fb[2][T::TN];
    auto read = [&](int st, int s) {
#pragma unroll
        for (int j = 0; j < T::TN; ++j) fb[s][j] = *reinterpret_cast<const frag_t*>(smem + st * T::STAGE_BYTES + (get_b[j] ^ (s << 6)));
#pragma unroll
        for (int i = 0; i < T::TM; ++i) fa[s][i] = *reinterpret_cast<const frag_t*>(smem + st * T::STAGE_BYTES + (get_a[i] ^ (s << 6)));
    };
    auto multiply = [&](int s) {
#pragma unroll
        for (int i = 0; i < T::TM; ++i)
#pragma unroll
            for (int j = 0; j < T::TN; ++j) {
                if constexpr (T::F16) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[s][j], fa[s][i], acc[i][j], 0, 0, 0);
                else acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[s][j], fa[s][i], acc[i][j], 0, 0, 0);
            }
    };
    auto put = [&](int u) {
        la.store(ra[u], smem + u * T::STAGE_BYTES);
        lb.store(rb[u], smem + u * T::STAGE_BYTES + T::BM * kRowBytes);
    };
    auto fetch = [&](int u, int slab) {        // slabs behind the last one: operands of no extent, zeros without a memory access
        ProdOperand a = job.a, b = job.b;
        if (slab >= slabs) a.extent = b.extent = 0;
        la.load(a, slab, ra[u]);
        lb.load(b, slab, rb[u]);
    };
    // The slab lies in stage u, the fragments of its first half in registers.  The second half's are read and the next slab is
    // written under the first half's MFMAs; behind the barrier the next slab's first half is read under the second half's.
    // (One body for every slab: with bodies of their own for the last ones, which need not write and request, the compiler spills.)
    auto step = [&](auto U, int slab) {
        constexpr int u = decltype(U)::value;
        read(u, 1);
        multiply(0);
        put(u ^ 1);
        fetch(u ^ 1, slab + 1 + D);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        read(u ^ 1, 0);
        multiply(1);
    };
    fetch(0, 0);
    fetch(1, 1);
    put(0);
    fetch(0, D);
    __syncthreads();
    read(0, 0);
    int slab = 0;
    for (; slab + 2 <= slabs; slab += 2) {
        step(std::integral_constant<int, 0>{}, slab);
        step(std::integral_constant<int, 1>{}, slab + 1);
    }
    if (slab < slabs) step(std::integral_constant<int, 0>{}, slab);
}
// Tiles: job(id, j) the operands of tile `id` (false: no such tile), finish(id, acc, smem) its epilogue.
template <class T, class Tiles>
__device__ __forceinline__ void prod_tile(const Tiles& tiles, unsigned char* smem) {
    ProdJob job;
    if (!tiles.job(blockIdx.x, job)) return;
    job = ProdJob{prod_uniform(job.a), prod_uniform(job.b), __builtin_amdgcn_readfirstlane(job.slabs)};
    f32x4 acc[T::TM][T::TN];
    prod_slabs<T>(job, smem, acc);
    tiles.finish(blockIdx.x, acc, smem);
}

// What the epilogue of a tile without bias needs: rows of C from `c` on, N columns a row, this tile's from n0 on.
__device__ __forceinline__ TaskPtrs prod_epilogue(uint16_t* c, int N, int n0, int rows) {
    TaskPtrs p{};
    p.c_base = c;
    p.N = N;
    p.rows = rows;
    p.n0 = n0;
    p.act = MOE_ACT_NONE;
    return p;
}

// Weight gradient of one projection from the packed rows as they are: dw[e] [N, K] = sum over expert e's rows of
// dy[r, :]^T a[r, :].  Tiles expert by expert.  The workgroups of an XCD (launched eight apart) take neighbouring tiles, four
// columns wide, whose operands meet in its L2: 16 experts of 2048 x 1408, 750 rows each, 104 us against 124 with columns fastest.
// Up to three of them share a launch, a projection's tiles behind another's (a step's tiles need not fill whole rounds projection by
// projection, and the workgroups that stay fill and drain once).  Three launches / one, us: 4 experts of 2048 x 2560, 4096 rows each
// 532 / 406; 8 of 1536 x 1920, 512 rows 129 / 106; 8 of 1280 x 1664, 256 rows 79 / 58; 16 of 1152 x 1920, 175 rows 110 / 90; 16 of 2048 x
// 2048, 512 rows 277 / 256; of 2048 x 1408, 750 rows (whole rounds either way) 250 / 243.
struct WgradJob {
    const uint16_t* dy;
    const uint16_t* a;
    uint16_t* dw;
    int N, K;
};
template <class T>
struct WgradTiles {
    WgradJob p0, p1, p2;         // (selected by comparisons: an index that is not a constant would put them into scratch memory)
    const int32_t* count;
    const int32_t* offset;
    int E;
    // ids of one projection; a multiple of 8, so that an id's XCD does not depend on the projection
    static __host__ __device__ __forceinline__ int64_t ids(const WgradJob& p, int E) {
        return (int64_t)(((p.K + T::BN - 1) / T::BN * ((p.N + T::BM - 1) / T::BM) + 7) / 8 * 8) * E;
    }
    // Tile `id`: which projection, of which expert, from which row and column of its gradient on; false: no such tile.
    __device__ __forceinline__ bool place(int id, WgradJob& p, int& e, int& n0, int& k0) const {
        const int ids0 = (int)ids(p0, E), ids1 = ids0 + (int)ids(p1, E);
        const int which = id < ids0 ? 0 : id < ids1 ? 1 : 2;
        id -= which == 0 ? 0 : which == 1 ? ids0 : ids1;
        p.dy = which == 0 ? p0.dy : which == 1 ? p1.dy : p2.dy;
        p.a = which == 0 ? p0.a : which == 1 ? p1.a : p2.a;
        p.dw = which == 0 ? p0.dw : which == 1 ? p1.dw : p2.dw;
        p.N = which == 0 ? p0.N : which == 1 ? p1.N : p2.N;
        p.K = which == 0 ? p0.K : which == 1 ? p1.K : p2.K;
        const int cols = (p.K + T::BN - 1) / T::BN, rows = (p.N + T::BM - 1) / T::BM, share = (cols * rows + 7) / 8;
        if (cols * rows == 0) return false;
        e = id / (8 * share);
        const int r = id - e * 8 * share, t = (r & 7) * share + (r >> 3);
        const int band = t / (4 * rows), in = t - band * 4 * rows, width = min(4, cols - 4 * band);
        if (t >= cols * rows) return false;
        n0 = in / width * T::BM;
        k0 = (4 * band + in % width) * T::BN;
        return e < E;
    }
    __device__ __forceinline__ ProdJob operands(const WgradJob& p, int e, int n0, int k0) const {
        const int n = max(count[e], 0);
        const int64_t off = offset[e];
        ProdJob j;
        j.a = ProdOperand{p.dy + off * p.N + n0, p.N, n > 0 ? (uint32_t)(((int64_t)n * p.N - n0) * 2) : 0u};
        j.b = ProdOperand{p.a + off * p.K + k0, p.K, n > 0 ? (uint32_t)(((int64_t)n * p.K - k0) * 2) : 0u};
        j.slabs = max((n + kBK - 1) / kBK, 1);
        return j;
    }
    __device__ __forceinline__ TaskPtrs result(const WgradJob& p, int e, int n0, int k0) const {
        return prod_epilogue(p.dw + ((int64_t)e * p.N + n0) * p.K, p.K, k0, min(T::BM, p.N - n0));
    }
    __device__ __forceinline__ bool job(int id, ProdJob& j) const {
        WgradJob p;
        int e, n0, k0;
        if (!place(id, p, e, n0, k0)) return false;
        j = operands(p, e, n0, k0);
        return true;
    }
    __device__ __forceinline__ void finish(int id, f32x4 (&acc)[T::TM][T::TN], unsigned char* smem) const {
        WgradJob p;
        int e, n0, k0;
        place(id, p, e, n0, k0);
        grouped_epilogue<T, kSums>(result(p, e, n0, k0), smem, acc);
    }
};
template <class T>
__global__ __launch_bounds__(T::THREADS, 2) void wgrad_rows_kernel(WgradTiles<T> tiles) {
    extern __shared__ __align__(16) unsigned char smem[];
    prod_tile<T>(tiles, smem);
}

// The same on the hand-ordered 256 x 256 tile, both operands turned round by the fragment reads.  A tile's sum is short (8 slabs of 512
// rows are 11 us) against what surrounds it, so the workgroups stay: the next tile's first two slabs are on their way while this
// one's results are stored.  16 experts of 2048 x 2048, 512 rows each: a workgroup per tile 87 us, this 81 (the 128 x 128 tiles 101);
// of 2048 x 1408, 750 rows 81 and 82 (96); 4 of 2048 x 2560, 4096 rows 174 and 174 (192), 1.72 PFLOP/s inside the slab loop.
template <class T>
__global__ __launch_bounds__(T::THREADS) void wgrad_ring_kernel(WgradTiles<T> w, int ids) {
    extern __shared__ __align__(16) unsigned char smem[];
    auto find = [&](int id, TaskPtrs& p) {     // the first tile from `id` on, in steps of the grid
        WgradJob of;
        int e, n0, k0;
        while (id < ids && !w.place(id, of, e, n0, k0)) id += gridDim.x;
        if (id >= ids) return id;
        const ProdJob j = w.operands(of, e, n0, k0);
        p = w.result(of, e, n0, k0);
        p.a_base = j.a.base;
        p.a_ld = j.a.ld;
        p.a_extent = j.a.extent;
        p.b0 = j.b.base;
        p.b_ld = j.b.ld;
        p.b_extent = j.b.extent;
        p.K = j.slabs * kBK;
        return id;
    };
    TaskPtrs p;
    int id = find(blockIdx.x, p);
    if (id >= ids) return;
    RingLoads L = ring_prepare<T>(p);
    ring_first_loads<T>(L, smem);
    while (true) {
        f32x4 acc[T::TM][T::TN];
        const bool mine = ring_slabs<T>(p.rows, L, smem, acc);
        __builtin_amdgcn_s_barrier();          // every wavefront has read its last fragments (ring_slabs waits for them)
        TaskPtrs next;
        id = find(id + gridDim.x, next);
        if (id < ids) {
            L = ring_prepare<T>(next);
            ring_first_loads<T>(L, smem);
        }
        if (mine) grouped_epilogue<T, kSums>(p, smem, acc);
        if (id >= ids) return;
        p = next;
    }
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
// Tile of one grouped product (or of `products` that share a launch), as for a layer: 1, 2, or 0 when an operand has 4 GiB or more.
int grouped_gemm_tile_16(int64_t A, int E, int N, int K, int products) {
    if (!grouped_hand_ok(A, N, K)) return 0;
    const int e = E > 0 ? E : 1, cols = products * columns256(N);
    return projection_cost(true, A, e, cols, K) <= projection_cost(false, A, e, cols, K) ? 1 : 2;
}

template <class P, int EPI>
static hipError_t launch_grouped(const GroupedArgs& g, int64_t A, hipStream_t st) {
    const auto kernel = &grouped_gemm_kernel<P, EPI>;
    hipError_t e = allow_lds(kernel, P::LDS_BYTES);
    if (e != hipSuccess) return e;
    constexpr int COLS = EPI == kSwiglu ? P::BN / 2 : P::BN;
    const int64_t cols = (int64_t)((g.N + COLS - 1) / COLS) * (EPI == kSums && g.out1 ? 2 : 1);
    const int64_t blocks = (A / P::BIG + g.E) * cols + kShareSlack;      // no expert has more than rows / BIG + 1 row blocks
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

// out = a_rows . w[e]^T and out1 = a_rows . w1[e]^T in one launch; tile: 1 or 2.
hipError_t launch_grouped_gemm_pair_16(const void* a_rows, const void* w, const void* w1, void* out, void* out1, const int32_t* count,
                                       const int32_t* offset, int tile, int64_t A, int E, int N, int K, bool f16, hipStream_t st) {
    const GroupedArgs g{(const uint16_t*)a_rows, (const uint16_t*)w, nullptr, nullptr, nullptr, (uint16_t*)out, (uint16_t*)out1,
                        count, offset, E, N, K, MOE_ACT_NONE, (uint32_t)(A * K * 2), nullptr, (const uint16_t*)w1, nullptr, (const uint16_t*)a_rows};
    return f16 ? launch_grouped_tile<true, kSums>(g, tile, A, st) : launch_grouped_tile<false, kSums>(g, tile, A, st);
}

// tile: 1 (256-row blocks), 2 (128-row blocks) or 0 (the 128 x 128 tile of the general loop).
hipError_t launch_grouped_gemm_16(const void* a_rows, const void* w, const void* bias, void* out, const int32_t* count,
                                  const int32_t* offset, int tile, int64_t A, int E, int N, int K, int act, bool f16, hipStream_t st) {
    const GroupedArgs g{(const uint16_t*)a_rows, (const uint16_t*)w, (const uint16_t*)bias, nullptr, nullptr, (uint16_t*)out, nullptr,
                        count, offset, E, N, K, act, (uint32_t)(A * K * 2), nullptr, nullptr, nullptr, nullptr};
    if (act == MOE_ACT_GELU) return f16 ? launch_grouped_tile<true, kGelu>(g, tile, A, st) : launch_grouped_tile<false, kGelu>(g, tile, A, st);
    return f16 ? launch_grouped_tile<true, kSums>(g, tile, A, st) : launch_grouped_tile<false, kSums>(g, tile, A, st);
}

// tile: 1 or 2: the hand-ordered tiles and those for their remainders only.
hipError_t launch_grouped_gemm_deriv_16(const void* a_rows, const void* w, const void* u, const void* g_rows, void* du, void* dg,
                                        const int32_t* count, const int32_t* offset, int tile, int64_t A, int E, int N, int K,
                                        int hidden_act, bool f16, hipStream_t st) {
    const GroupedArgs g{(const uint16_t*)a_rows, (const uint16_t*)w, nullptr, (const uint16_t*)u, (const uint16_t*)g_rows, (uint16_t*)du,
                        (uint16_t*)dg, count, offset, E, N, K, hidden_act, (uint32_t)(A * K * 2), nullptr, nullptr, nullptr, nullptr};
    return f16 ? launch_grouped_tile<true, kDeriv>(g, tile, A, st) : launch_grouped_tile<false, kDeriv>(g, tile, A, st);
}

// A layer's two projections, a launch each: blocks of 256 rows and the 128-row tile for what an expert has left, or blocks of 128 rows.
// Whole layers, us, the queue / two launches of it in the order of the row block table / this:
//   128-row blocks: 12 experts of 1344 x 2752, GELU, 150 rows each 122 / 108 / 107, 250 rows 130 / 118 / 115; 64 of 2048 x 1408, SwiGLU,
//   94 rows 294 / 306 / 282; 8 of 4096 x 14336, 128 rows 726 / 740 / 706; 16 of 2048 x 2048, 128 rows 130 / 113 / 109
//   256-row blocks, and which layers run so: two_launches.hpp
template <class P>
static hipError_t launch_ffn_split(const FfnArgs& a, const ExpertRows& rows, hipStream_t st) {
    const int64_t A = (int64_t)a.S * a.k;
    GroupedArgs g{(const uint16_t*)a.x, (const uint16_t*)a.w_up, (const uint16_t*)a.b_up, nullptr, nullptr, (uint16_t*)a.h, nullptr,
                  rows.count, rows.offset, a.E, a.I, a.H, a.act, a.x_bytes, a.token_indices, (const uint16_t*)a.w_gate, (const uint16_t*)a.b_gate, nullptr};
    const hipError_t e = a.act == MOE_ACT_SWIGLU ? launch_grouped<P, kSwiglu>(g, A, st)
                         : a.act == MOE_ACT_GELU ? launch_grouped<P, kGelu>(g, A, st) : launch_grouped<P, kSums>(g, A, st);
    if (e != hipSuccess) return e;
    g = GroupedArgs{(const uint16_t*)a.h, (const uint16_t*)a.w_down, (const uint16_t*)a.b_down, nullptr, nullptr, (uint16_t*)a.y, nullptr,
                    rows.count, rows.offset, a.E, a.H, a.I, MOE_ACT_NONE, a.h_bytes, nullptr, nullptr, nullptr, nullptr};
    return launch_grouped<P, kSums>(g, A, st);
}
static TwoLaunchShape two_launch_shape(const FfnArgs& a) { return TwoLaunchShape{(int64_t)a.S * a.k, a.E, a.H, a.I, a.act == MOE_ACT_SWIGLU}; }
bool ffn_split_16_keeps_table(const FfnArgs& a) { return two_launches_keep_table(two_launch_shape(a)); }
hipError_t launch_ffn_split_16(const FfnArgs& a, const ExpertRows& rows, int block_rows, bool f16, hipStream_t st) {
    if (block_rows == 128 && two_launches_on_256(two_launch_shape(a))) block_rows = 256;
    if (block_rows == 128) return f16 ? launch_ffn_split<RowSplit<true, 128>>(a, rows, st) : launch_ffn_split<RowSplit<false, 128>>(a, rows, st);
    return f16 ? launch_ffn_split<RowSplit<true, 256>>(a, rows, st) : launch_ffn_split<RowSplit<false, 256>>(a, rows, st);
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
    if (wgrad_hand_ok(N, K, ld))
        return f16 ? launch_wgrad<Tile256H>(dyT, aT, dw, poff, E, N, K, ld, st) : launch_wgrad<Tile256>(dyT, aT, dw, poff, E, N, K, ld, st);
    return f16 ? launch_wgrad<Tile128H>(dyT, aT, dw, poff, E, N, K, ld, st)
               : launch_wgrad<Tile128>(dyT, aT, dw, poff, E, N, K, ld, st);
}

template <class T>
static hipError_t launch_wgrad_rows(const WgradTiles<T>& w, hipStream_t st) {
    const int64_t tiles = WgradTiles<T>::ids(w.p0, w.E) + WgradTiles<T>::ids(w.p1, w.E) + WgradTiles<T>::ids(w.p2, w.E);
    if (tiles > INT32_MAX) return hipErrorInvalidValue;
    if constexpr (T::TRA) {
        hipError_t e = allow_lds(&wgrad_ring_kernel<T>, T::LDS_BYTES);
        if (e != hipSuccess) return e;
        wgrad_ring_kernel<T><<<(unsigned)std::min<int64_t>(tiles, kTaskUnits), T::THREADS, T::LDS_BYTES, st>>>(w, (int)tiles);
    } else {
        hipError_t e = allow_lds(&wgrad_rows_kernel<T>, T::LDS_BYTES);
        if (e != hipSuccess) return e;
        wgrad_rows_kernel<T><<<(unsigned)tiles, T::THREADS, T::LDS_BYTES, st>>>(w);
    }
    return hipGetLastError();
}
template <bool F16>
static hipError_t launch_wgrad_rows(const WgradOperands* ops, int n, const int32_t* count, const int32_t* offset, bool large, int E, hipStream_t st) {
    using Large = Tile<256, 256, 2, 2, 2, F16, true, true>;
    auto job = [&](int i) {
        return i < n ? WgradJob{(const uint16_t*)ops[i].dy, (const uint16_t*)ops[i].a, (uint16_t*)ops[i].dw, ops[i].N, ops[i].K} : WgradJob{};
    };
    if (large) return launch_wgrad_rows(WgradTiles<Large>{job(0), job(1), job(2), count, offset, E}, st);
    return launch_wgrad_rows(WgradTiles<ProdTile<F16>>{job(0), job(1), job(2), count, offset, E}, st);
}
// n weight gradients (1 to 3) in one launch; large: on the 256 x 256 tile.
hipError_t launch_wgrad_rows_16(const WgradOperands* ops, int n, const int32_t* count, const int32_t* offset, bool large, int E, bool f16, hipStream_t st) {
    return f16 ? launch_wgrad_rows<true>(ops, n, count, offset, large, E, st) : launch_wgrad_rows<false>(ops, n, count, offset, large, E, st);
}

template <bool F16, int EPI>
static hipError_t launch_grouped_kn(const GroupedArgs& g, bool large, int64_t A, hipStream_t st) {
    return large ? launch_grouped<RowSplit<F16, 256, true>, EPI>(g, A, st) : launch_grouped<RowSplit<F16, 128, true>, EPI>(g, A, st);
}
// out = a . w[e], or, with u, du (and dg) = (a . w[e]) * act'(u, g); large: on 256-row blocks and remainders.
hipError_t launch_grouped_gemm_kn_16(const void* a_rows, const void* w, const void* u, const void* g_rows, void* out, void* out1,
                                     const int32_t* count, const int32_t* offset, bool large, int64_t A, int E, int N, int K, int hidden_act, bool f16,
                                     hipStream_t st) {
    const GroupedArgs g{(const uint16_t*)a_rows, (const uint16_t*)w, nullptr, (const uint16_t*)u, (const uint16_t*)g_rows, (uint16_t*)out,
                        (uint16_t*)out1, count, offset, E, N, K, u ? hidden_act : MOE_ACT_NONE, (uint32_t)(A * K * 2), nullptr, nullptr, nullptr, nullptr};
    if (u) return f16 ? launch_grouped_kn<true, kDeriv>(g, large, A, st) : launch_grouped_kn<false, kDeriv>(g, large, A, st);
    return f16 ? launch_grouped_kn<true, kSums>(g, large, A, st) : launch_grouped_kn<false, kSums>(g, large, A, st);
}
// out = a . w[e] and out1 = a1 . w1[e] in one launch.
hipError_t launch_grouped_gemm_kn_pair_16(const void* a_rows, const void* a1_rows, const void* w, const void* w1, void* out, void* out1,
                                          const int32_t* count, const int32_t* offset, bool large, int64_t A, int E, int N, int K, bool f16, hipStream_t st) {
    const GroupedArgs g{(const uint16_t*)a_rows, (const uint16_t*)w, nullptr, nullptr, nullptr, (uint16_t*)out, (uint16_t*)out1,
                        count, offset, E, N, K, MOE_ACT_NONE, (uint32_t)(A * K * 2), nullptr, (const uint16_t*)w1, nullptr, (const uint16_t*)a1_rows};
    return f16 ? launch_grouped_kn<true, kSums>(g, large, A, st) : launch_grouped_kn<false, kSums>(g, large, A, st);
}

}  // namespace moe355
