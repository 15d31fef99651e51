// Expert FFN of bf16 / fp16 layers on the MFMA tiles (ffn_bf16_tile.hpp): two launches, or one persistent kernel on the task queues.
#include "ffn_bf16_tile.hpp"

namespace moe355 {
namespace {

template <class T>
__device__ __forceinline__ TaskPtrs resolve(const FfnArgs& a, const Task& t, bool publish) {
    TaskPtrs p;
    const int64_t HI = (int64_t)a.H * a.I;
    const bool sw = a.act == MOE_ACT_SWIGLU;
    if (t.phase == 0) {
        p.a_base = (const uint16_t*)a.x;
        p.gather = a.token_indices + t.row0;
        p.a_row0 = 0;
        p.a_ld = a.H;
        p.b0 = (const uint16_t*)a.w_up + t.expert * HI;
        p.b1 = sw ? (const uint16_t*)a.w_gate + t.expert * HI : nullptr;
        p.bias0 = a.b_up ? (const uint16_t*)a.b_up + (int64_t)t.expert * a.I : nullptr;
        p.bias1 = (sw && a.b_gate) ? (const uint16_t*)a.b_gate + (int64_t)t.expert * a.I : nullptr;
        p.c_base = (uint16_t*)a.h + (int64_t)t.row0 * a.I;
        p.N = a.I;
        p.K = a.H;
        p.b_ld = a.H;
        p.n0 = t.ntile * (sw ? T::BN / 2 : T::BN);
        p.act = a.act;
        p.swiglu = sw;
        p.publish = publish;
    } else {
        p.a_base = (const uint16_t*)a.h;
        p.gather = nullptr;
        p.a_row0 = t.row0;
        p.a_ld = a.I;
        p.b0 = (const uint16_t*)a.w_down + t.expert * HI;
        p.b1 = nullptr;
        p.bias0 = a.b_down ? (const uint16_t*)a.b_down + (int64_t)t.expert * a.H : nullptr;
        p.bias1 = nullptr;
        p.c_base = (uint16_t*)a.y + (int64_t)t.row0 * a.H;
        p.N = a.H;
        p.K = a.I;
        p.b_ld = a.I;
        p.n0 = t.ntile * T::BN;
        p.act = MOE_ACT_NONE;
        p.swiglu = false;
        p.publish = publish;
    }
    p.rows = t.rows;
    p.a_extent = t.phase == 0 ? a.x_bytes : a.h_bytes;
    p.b_extent = a.w_bytes;
    p.part = nullptr;
    p.part_cnt = nullptr;
    p.kparts = 1;
    p.kpart = 0;
    p.poison = false;
    p.deriv = 0;
    p.aux0 = nullptr;
    p.aux1 = nullptr;
    p.c1_base = nullptr;
    if (t.phase == 1 && t.kparts > 1) {       // one of kparts partial sums: this part's share of the intermediate dimension
        const int Kp = a.I / t.kparts, k0 = t.kpart * Kp;
        p.K = Kp;
        p.a_base += k0;
        p.b0 += k0;
        p.a_extent -= (uint32_t)k0 * 2;       // the descriptors start where the operands now start
        p.b_extent -= (uint32_t)k0 * 2;
        const int tile = (t.mtile - a.q->split_mt0) * a.nnt1 + t.ntile;
        p.part = a.split_part + (size_t)tile * t.kparts * ((size_t)T::BM * T::BN);
        p.part_cnt = a.split_cnt + tile;
        p.kparts = t.kparts;
        p.kpart = t.kpart;
        p.poison = t.poison;
    }
    return p;
}

// A plan pairs the tile of the up(/gate) projection with the tile of the down projection; both use the
// same row-block height and the same workgroup size.
//
// TS (optional): the tile that takes the row blocks of at most TS::BM rows -- the ragged last block of an expert --
// in place of T0 / T1.  It covers the same columns per task, so the task tables do not change; it only does not
// spend a full tile's MFMAs on rows that are mostly padding.
template <class T0_, class T1_, class TS_ = void>
struct Plan {
    using T0 = T0_;
    using T1 = T1_;
    using TS = TS_;
    static constexpr bool MIXED = !std::is_void<TS_>::value;
    static_assert(T0::BM == T1::BM && T0::THREADS == T1::THREADS, "phases share row blocks and workgroup size");
    static constexpr int THREADS = T0::THREADS;
    static constexpr int LDS_BYTES = T0::LDS_BYTES > T1::LDS_BYTES ? T0::LDS_BYTES : T1::LDS_BYTES;
};
using LargePlan = Plan<Tile256, Tile256>;
using MixedPlan = Plan<Tile256, Tile256, Tile128x256>;
using MediumPlan = Plan<Tile128x256, Tile128x256>;
using SmallPlan = Plan<Tile128, Tile128>;
using LargePlanH = Plan<Tile256H, Tile256H>;
using MixedPlanH = Plan<Tile256H, Tile256H, Tile128x256H>;
using MediumPlanH = Plan<Tile128x256H, Tile128x256H>;
using SmallPlanH = Plan<Tile128H, Tile128H>;

// One task of a plan: the plan's tile, or its small-row-block tile when the block has few enough rows.
// SPLIT: the task may be a part of a tile (kernels of their own: the code for it costs the others 1-2 % in short tasks).
template <class P, bool SPLIT = false>
__device__ __forceinline__ void plan_tile(const FfnArgs& a, const Task& t, bool publish, unsigned char* smem) {
    static_assert(std::is_same<typename P::T0, typename P::T1>::value, "one tile for both projections: one inlined copy");
    const TaskPtrs p = resolve<typename P::T0>(a, t, publish);
    if constexpr (P::MIXED) {
        static_assert(P::TS::BN == P::T0::BN && P::TS::LDS_BYTES <= P::LDS_BYTES, "same columns per task");
        if (t.rows <= P::TS::BM) {
            if constexpr (SPLIT && P::TS::HAND) {
                if (p.part) {
                    gemm_tile_ring_part<typename P::TS>(p, smem);
                    return;
                }
            }
            gemm_tile<typename P::TS>(p, smem);
            return;
        }
    }
    if constexpr (SPLIT && P::T0::HAND) {
        if (p.part) {
            gemm_tile_ring_part<typename P::T0>(p, smem);
            return;
        }
    }
    gemm_tile<typename P::T0>(p, smem);
}

// One launch per phase; workgroup b runs task b of that phase.
template <class P, bool SPLIT = false>
__global__ __launch_bounds__(P::THREADS) void ffn_tiled_kernel(FfnArgs a, int phase) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_list[1 + P::T0::BM];
    using ET = typename std::conditional<P::T0::F16, f16_s, bf16_s>::type;
    if (phase == 0) zero_unrouted_rows(a, 2);
    Task t;
    if (!tiled_task(a, phase, blockIdx.x, t)) return;
    plan_tile<P, SPLIT>(a, t, phase == 1 && a.arrive, smem);   // rows another workgroup may combine go out write-through
    if (phase == 1 && a.arrive) combine_arrivals<ET>(combine_args(a), t.row0, t.rows, t.ntile, t.ntile * P::T1::BN, P::T1::BN, s_list);
}

// The kernel's argument block, read again from the kernel-argument segment through a pointer the compiler cannot see
// through: values loaded from it live only as long as they are used, instead of occupying forty scalar registers
// across the slab loop (which then spill into vector registers and bring vector instructions into the loop).
__device__ __forceinline__ const FfnArgs& kernel_args_again() {
    typedef const __attribute__((address_space(4))) FfnArgs* args_ptr;
    args_ptr q = (args_ptr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(q));
    return *(const FfnArgs*)q;
}

// Persistent workgroups popping (expert, tile) tasks from the queue of their XCD (protocol: ffn_common.hpp).
template <class P, bool SPLIT = false>
__global__ __launch_bounds__(P::THREADS) void ffn_persistent_kernel(FfnArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_task, s_ok;
    __shared__ int s_list[1 + P::T0::BM];
    static_assert(1 + P::T0::BM >= kCombineLds, "s_list doubles as the scratch of the combine tasks");
    using ET = typename std::conditional<P::T0::F16, f16_s, bf16_s>::type;
    queue_kernel_entry();
    queue_clock_stamp(kernel_args_again().wg_clock, 0);
    zero_unrouted_rows(kernel_args_again(), 2);
    const int ids = a.q->ids_queue;
    const int nseg = a.q->nseg;
    const int nnt0 = a.seg_phase0[0].nnt;
    QueueCursor cur = queue_cursor(a.groups);
    Task t;
    while (next_task(a, cur, &s_task, ids, nseg, nnt0, t)) {   // uniform exit: every wavefront leaves together
        if (t.phase == 1 && !wait_phase0_done(a.done0, t.mtile, nnt0, a.spin_limit, a.q, a.host_stall, &s_ok)) {
            // the rows never became ready: NaN instead of a result, and a tile of no rows (it loads, computes and
            // stores nothing of its own), so that the loop keeps its one shape; a part of a tile keeps its shape too (the
            // parts must agree on it) and hands on NaN in place of its sums
            if (t.kparts > 1) {
                t.poison = true;
            } else {
                poison_tile((uint16_t*)a.y + (int64_t)t.row0 * a.H, t.rows, a.H, t.ntile * P::T1::BN, P::T1::BN, 2);
                t.rows = 0;
            }
        }
        const long long started = trace_clock(kernel_args_again().task_trace);
        plan_tile<P, SPLIT>(a, t, t.phase == 0 || publish_y(a), smem);
        if (kernel_args_again().task_trace)
            trace_task(kernel_args_again().task_trace, kernel_args_again().task_trace_cap, t.phase | (t.kparts > 1 ? (t.kpart << 2) | (t.kparts << 4) : 0), t.expert, t.mtile, t.ntile, t.rows, started);
        if (t.phase == 0) signal_phase0_done(a.done0, t.mtile);
        else                 // the row count from the table: a tile whose wait expired runs with none, and still arrives
            after_down_tile<ET>(kernel_args_again(), t.row0, a.mtiles[t.mtile].rows, t.mtile, t.ntile, t.ntile * P::T1::BN, P::T1::BN, s_list);
    }
    if (kernel_args_again().combined) combine_while_idle<ET>(sweep_args(kernel_args_again()), &s_task, s_list);
    queue_clock_stamp(kernel_args_again().wg_clock, 1);
}

// The same queue for the 256 x 256 tile, with the start of the next task moved under the end of the current one
// (opt-in: option queue_early = 1).
//
// Between two tiles a workgroup pops (an atomic round trip and two barriers), decodes, computes its row offsets (eight
// gathered token indices per thread), issues the first 32 loads and waits for slab 0.  Here the next id is reserved
// with an asynchronous pop when the current tile's slab loop begins (its latency disappears under the loop), and right
// behind the loop -- the LDS stages are free, the accumulators still hold the tile -- the next task is decoded, its
// dependency polled once, the weight rows of its first two slabs are requested, and the token rows follow two at a
// time between the row groups of the current tile's epilogue.  A next task that cannot start (dependency not yet
// met, queue exhausted, a hole) is handled after the epilogue the plain way; a workgroup never blocks while it holds
// unstored results, so the queue's progress argument is unchanged.  Near the end of its queue a workgroup stops
// reserving: a task reserved behind a long tile would start late while other workgroups idle.
// Measured with timestamps inside the kernel (Mixtral shape, per tile): the wait for slab 0 (about 4 us) is gone, but
// pop result + barrier 0.8, decode 1.2, offsets 1.2 and issuing the loads 1.4 us now sit in front of the epilogue, so
// the time between two slab loops stays at 12-13 us and the launch takes the same number of cycles (MFMA pipes busy
// 74 % either way); short tiles lose 2-3 %.  Results are bit-identical to the plain loop.
constexpr int kReserveMargin = 64;   // ids left in the current queue below which tasks are popped late again

template <class P>
__global__ __launch_bounds__(P::THREADS) void ffn_persistent_ring_kernel(FfnArgs) {
    using T = typename P::T0;
    static_assert(std::is_same<typename P::T0, typename P::T1>::value && T::RING, "the hand-ordered tile for both projections");
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_task, s_ok, s_next[2];
    __shared__ int s_list[1 + T::BM];
    using ET = typename std::conditional<T::F16, f16_s, bf16_s>::type;
    queue_kernel_entry();
    queue_clock_stamp(kernel_args_again().wg_clock, 0);
    zero_unrouted_rows(kernel_args_again(), 2);
    int ids, nseg, nnt0, groups;
    {
        const FfnArgs& a = kernel_args_again();
        ids = a.q->ids_queue;
        nseg = a.q->nseg;
        nnt0 = a.seg_phase0[0].nnt;
        groups = a.groups;
    }
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    QueueCursor cur = queue_cursor(groups);
    // The current task as plain scalars (a struct carried around the loop ends up in scratch memory).
    int ph = 0, ex = 0, mt = 0, nt = 0, row0 = 0, rows = 0;
    auto as_task = [&]() {
        Task q;
        q.phase = ph; q.expert = ex; q.mtile = mt; q.ntile = nt; q.row0 = row0; q.rows = rows; q.nnt0 = nnt0; q.valid = true;
        q.kparts = 1; q.kpart = 0; q.poison = false;     // (the host never asks for this loop and partial sums together)
        return q;
    };
    RingLoads L;
    // a task started the plain way: wait for its rows if need be, offsets, first loads
    auto start_cold = [&]() {
        const FfnArgs& a = kernel_args_again();
        if (ph == 1 && !wait_phase0_done(a.done0, mt, nnt0, a.spin_limit, a.q, a.host_stall, &s_ok)) {
            poison_tile((uint16_t*)a.y + (int64_t)row0 * a.H, rows, a.H, nt * T::BN, T::BN, 2);
            rows = 0;
        }
        L = ring_prepare<T>(resolve<T>(a, as_task(), ph == 0));
        __syncthreads();                        // the previous task may still be reading the stages
        ring_first_loads<T>(L, smem);
    };
    auto pop_blocking = [&]() {
        Task q;
        const bool ok = next_task(kernel_args_again(), cur, &s_task, ids, nseg, nnt0, q);
        if (ok) { ph = q.phase; ex = q.expert; mt = q.mtile; nt = q.ntile; row0 = q.row0; rows = q.rows; }
        return ok;
    };
    bool have = pop_blocking();
    if (have) start_cold();
    while (have) {                              // uniform: every wavefront takes the same turns
        const bool reserve = cur.last_id + kReserveMargin < ids;
        int rid = 0;
        if (reserve && wave == 0) rid = pop_async(&kernel_args_again().q->heads[cur.group]);
        const long long traced_from = trace_clock(kernel_args_again().task_trace);   // the first loads left earlier, under the previous tile's end
        f32x4 acc[8][8];
        const bool active = ring_slabs<T>(rows, L, smem, acc);

        const FfnArgs& a = kernel_args_again();
        int nid = ids, n_valid = 0, n_ph = 0, n_ex = 0, n_mt = 0, n_nt = 0, n_row0 = 0, n_rows = 0, started = 0;
        if (reserve) {
            if (wave == 0) s_next[0] = pop_async_result(rid);
            __syncthreads();                    // also: every wavefront is done with the stages
            nid = __builtin_amdgcn_readfirstlane(s_next[0]);
            if (nid < ids) {
                const Task q = decode_task(a.seg_queue, nseg, a.mtiles, nid, cur.group, groups, nnt0, a.row_chunk);
                n_valid = q.valid; n_ph = q.phase; n_ex = q.expert; n_mt = q.mtile; n_nt = q.ntile; n_row0 = q.row0; n_rows = q.rows;
                if (n_valid) {
                    int ready = 1;
                    if (n_ph == 1) {            // one look at the dependency; the answer must be the workgroup's, not a wavefront's
                        if (wave == 0)
                            s_next[1] = __hip_atomic_load(a.done0 + n_mt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= nnt0;
                        __syncthreads();
                        ready = __builtin_amdgcn_readfirstlane(s_next[1]);
                        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
                    }
                    if (ready) {                // the loop is done with the old offsets
                        const TaskPtrs pq = resolve<T>(a, q, n_ph == 0);
                        L = ring_prepare_weights<T>(pq);
                        ring_first_weight_loads<T>(L, smem);
                        ring_prepare_tokens<T>(pq, L);
                        started = 1;
                    }
                }
            }
        }
        // the token rows of the next task's first slabs leave two at a time under the epilogue's arithmetic
        auto token_loads = [&](int i) {
            if (started) {
                ring_first_token_load<T>(L, smem, 2 * i);
                ring_first_token_load<T>(L, smem, 2 * i + 1);
            }
        };
        if (active) {
            epilogue_full_n<T>(resolve<T>(a, as_task(), ph == 0 || publish_y(a)), smem, acc, token_loads);
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) token_loads(i);
        }
        if (a.task_trace) trace_task(a.task_trace, a.task_trace_cap, ph, ex, mt, nt, rows, traced_from);
        if (ph == 0) signal_phase0_done(a.done0, mt);
        else after_down_tile<ET>(a, row0, a.mtiles[mt].rows, mt, nt, nt * T::BN, T::BN, s_list);
        if (reserve && nid < ids && n_valid) {   // the reserved task is the next one
            ph = n_ph; ex = n_ex; mt = n_mt; nt = n_nt; row0 = n_row0; rows = n_rows;
            cur.last_id = nid;
            if (!started) start_cold();          // its rows were not ready: wait now that nothing unstored is held
            continue;
        }
        if (reserve && nid >= ids) {             // the reserved pop found this queue empty: move on as next_task does
            if (++cur.exhausted >= groups) break;
            cur.group = cur.group + 1 == groups ? 0 : cur.group + 1;
        }
        have = pop_blocking();
        if (have) start_cold();
    }
    if (kernel_args_again().combined) combine_while_idle<ET>(sweep_args(kernel_args_again()), &s_task, s_list);
    queue_clock_stamp(kernel_args_again().wg_clock, 1);
}

template <class P>
hipError_t launch_tiled(const FfnArgs& a, int max_mtiles, int nnt0, int nnt1, hipStream_t st) {
    hipError_t e = allow_lds(&ffn_tiled_kernel<P>, P::LDS_BYTES);
    if (e != hipSuccess) return e;
    ffn_tiled_kernel<P><<<tiled_grid(max_mtiles, nnt0, a.groups), P::THREADS, P::LDS_BYTES, st>>>(a, 0);
    if constexpr (P::T0::HAND) {
        if (a.split_cnt) {      // row blocks whose tiles run as partial sums count once per part
            e = allow_lds(&ffn_tiled_kernel<P, true>, P::LDS_BYTES);
            if (e != hipSuccess) return e;
            ffn_tiled_kernel<P, true><<<tiled_grid(max_mtiles + a.split_extra_blocks, nnt1, a.groups), P::THREADS, P::LDS_BYTES, st>>>(a, 1);
            return hipGetLastError();
        }
    }
    ffn_tiled_kernel<P><<<tiled_grid(max_mtiles, nnt1, a.groups), P::THREADS, P::LDS_BYTES, st>>>(a, 1);
    return hipGetLastError();
}

template <class P>
hipError_t launch_persistent(const FfnArgs& a, int blocks, bool early, hipStream_t st) {
    if constexpr (P::T0::RING && !P::MIXED) {
        // option queue_early: the queue loop that starts the next task under the end of the current one (measured: no
        // faster on the Mixtral shape, 2-3 % slower on short tiles; kept for machines where the balance differs)
        if (early) {
            hipError_t e = allow_lds(&ffn_persistent_ring_kernel<P>, P::LDS_BYTES);
            if (e != hipSuccess) return e;
            ffn_persistent_ring_kernel<P><<<blocks, P::THREADS, P::LDS_BYTES, st>>>(a);
            return hipGetLastError();
        }
    }
    if constexpr (P::T0::HAND) {
        if (a.split_cnt) {
            hipError_t e = allow_lds(&ffn_persistent_kernel<P, true>, P::LDS_BYTES);
            if (e != hipSuccess) return e;
            ffn_persistent_kernel<P, true><<<blocks, P::THREADS, P::LDS_BYTES, st>>>(a);
            return hipGetLastError();
        }
    }
    hipError_t e = allow_lds(&ffn_persistent_kernel<P>, P::LDS_BYTES);
    if (e != hipSuccess) return e;
    ffn_persistent_kernel<P><<<blocks, P::THREADS, P::LDS_BYTES, st>>>(a);
    return hipGetLastError();
}

template <class P>
int occupancy() {
    int n = 0;
    if (allow_lds(&ffn_persistent_kernel<P>, P::LDS_BYTES) != hipSuccess) return 1;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void*>(&ffn_persistent_kernel<P>),
                                                     P::THREADS, P::LDS_BYTES) != hipSuccess || n < 1)
        n = 1;
    return n;
}

}  // namespace

static bool large_tile_ok(int64_t pairs, int H, int I) {
    return pairs * H * 2 < kBufferLimit && pairs * I * 2 < kBufferLimit && hand_weights_ok(H, I) && hand_weights_ok(I, H);
}

// The weight streamer's form for this many rows per expert, or -1: the tiles are faster.  The first line lies where too many
// experts begin to have a second block of 16 rows, the second where the tiles' cost, which rows do not change below a row
// block, is that of the streamer's token rows: both sides measured at 2 to 32 rows, figures in ffn_stream16.hip, for uneven routing as well.
static int stream16_form(int64_t pairs, int experts) {
    const double rows = (double)pairs / experts;
    return rows <= 9 ? 0 : rows <= 17 ? 1 : -1;
}

// Tile of a layer: 0 = 128 x 128 on the general loop (operands of 4 GiB and more), 1 = 256 x 256, 2 = 128 x 256,
// 3 = 256 x 256 with the 128 x 256 tile for the row blocks of at most 128 rows (option tile16 only), kStream16Tile + form =
// the weight streamer (ffn_stream16.hip; no option names it).
int bf16_tile(int64_t pairs, int experts, int H, int I, int swiglu, int opt_block_rows, int opt_tile) {
    if (!large_tile_ok(pairs, H, I)) return 0;
    // option block_rows: 256 means the 256 x 256 tile where it is not ragged in either projection ...
    if (opt_block_rows == 128 || opt_block_rows == 256)
        return opt_block_rows == 256 && H % 256 == 0 && I % (swiglu ? 128 : 256) == 0 ? 1 : 0;
    if (opt_tile >= 0 && opt_tile <= 3) return opt_tile;      // ... or tile16
    const int E = experts > 0 ? experts : 1;
    const int form = stream16_form(pairs, E);
    if (form >= 0) return kStream16Tile + form;
    auto cost = [&](bool large) {
        return projection_cost(large, pairs, E, columns256(swiglu ? 2 * I : I), H) + projection_cost(large, pairs, E, columns256(H), I);
    };
    return cost(true) <= cost(false) ? 1 : 2;
}
int bf16_block_m(int tile) {
    if (tile >= kStream16Tile) return stream16_block_m(tile - kStream16Tile);
    return tile == 1 || tile == 3 ? 256 : 128;
}
// Weight rows of a task: with SwiGLU half of them are gate rows (the streamer's tasks have as many columns either way).
int bf16_block_n0(int tile, int swiglu) {
    if (tile >= kStream16Tile) return stream16_block_n(tile - kStream16Tile) * (swiglu ? 2 : 1);
    return tile == 0 ? SmallPlan::T0::BN : 256;
}
int bf16_block_n1(int tile) {
    if (tile >= kStream16Tile) return stream16_block_n(tile - kStream16Tile);
    return tile == 0 ? SmallPlan::T1::BN : 256;
}

template <template <class> class F, class... Args>
static auto for_plan(int tile, bool f16, Args&&... args) {
    if (f16) {
        if (tile == 1) return F<LargePlanH>::run(args...);
        if (tile == 3) return F<MixedPlanH>::run(args...);
        if (tile == 2) return F<MediumPlanH>::run(args...);
        return F<SmallPlanH>::run(args...);
    }
    if (tile == 1) return F<LargePlan>::run(args...);
    if (tile == 3) return F<MixedPlan>::run(args...);
    if (tile == 2) return F<MediumPlan>::run(args...);
    return F<SmallPlan>::run(args...);
}
template <class P> struct RunTiled {
    static hipError_t run(const FfnArgs& a, int max_mtiles, int nnt0, int nnt1, hipStream_t st) { return launch_tiled<P>(a, max_mtiles, nnt0, nnt1, st); }
};
template <class P> struct RunPersistent {
    static hipError_t run(const FfnArgs& a, int blocks, bool early, hipStream_t st) { return launch_persistent<P>(a, blocks, early, st); }
};
template <class P> struct RunOccupancy {
    static int run() { return occupancy<P>(); }
};

hipError_t launch_ffn_tiled_bf16(const FfnArgs& a, const ExpertRows& rows, int tile, int max_mtiles, int nnt0, int nnt1,
                                 hipStream_t st, bool f16) {
    if (tile >= kStream16Tile) return launch_ffn_stream16(a, tile - kStream16Tile, f16, max_mtiles, nnt0, nnt1, 0, st);
    // (the combine inside the FFN kernels, partial sums and orders of the table: options, which the kernels on the row block table take)
    if (tile >= 1 && tile <= 3 && rows.count && !a.arrive && !a.split_cnt && !(tile == 1 && ffn_split_16_keeps_table(a))) return launch_ffn_split_16(a, rows, bf16_block_m(tile), f16, st);
    return for_plan<RunTiled>(tile, f16, a, max_mtiles, nnt0, nnt1, st);
}

hipError_t launch_ffn_persistent_bf16(const FfnArgs& a, int tile, int blocks, bool early, hipStream_t st, bool f16) {
    if (tile >= kStream16Tile) return launch_ffn_stream16(a, tile - kStream16Tile, f16, 0, 0, 0, blocks, st);
    return for_plan<RunPersistent>(tile, f16, a, blocks, early, st);
}

int ffn_persistent_occupancy_bf16(int tile) {
    if (tile >= kStream16Tile) return ffn_persistent_occupancy_stream16(tile - kStream16Tile);
    return for_plan<RunOccupancy>(tile, false);
}

}  // namespace moe355
