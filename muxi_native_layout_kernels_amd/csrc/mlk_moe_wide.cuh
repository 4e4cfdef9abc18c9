// Fused MoE for prefill-sized batches on the eight-wave panel loop (mlk_panel8.cuh): all tokens of a pass go through the
// two grouped products at once, so that every expert's weights are streamed once per pass.
//
//   gate/up   panel = 128 columns of the intermediate (128 gate rows and the 128 up rows with the same index, dealt to
//             the four row quarters of the panel as 32 + 32, so that gate and up of an element sit in the same
//             accumulator slot of one wave) x the up to 256 routed tokens of a task.  SiLU(gate) * up goes to the
//             intermediate, row-major [slot][I], turned around in LDS so that whole lines are stored.
//   down      panel = 256 output rows x the same task over one K slice; products times the routing weight go to an fp32
//             buffer [routed pair][K slice][H] for moe_combine_kernel, which adds them per token in pick order.
//
// A task holds up to 16 blocks of 16 routed tokens of one expert; an expert with more is split into tasks of nearly equal
// size in units of 64 tokens (moe_align_kernel), and a panel multiplies 64, 128, 192 or 256 token columns, whichever covers
// its task: with 512 +- 20 tokens per expert (2048 tokens, 8 experts, top-2) tasks filled to 256 first would leave a third,
// nearly empty panel for half of the experts.
//
// Order of the work: the (expert, row tile, task of the expert) triples, tasks fastest, form one line that is cut into
// eight equal runs, one per XCD (workgroup id modulo 8).  The tasks of an expert that share a row tile's weights then run
// next to each other on one L2, and an XCD works on few experts at a time, so its token rows stay there too.  Equal runs are unequal
// work where tasks differ in width; there one workgroup per CU fetches its items from queues (wide_queue_pays).  One workgroup per
// item -> queues, 8 experts, top-2, H 4096, I 14336, whole layer: bf16 658 -> 606 us at 420 tokens, 1079 -> 963 at 1100,
// 1587 -> 1529 at 2048; soft-FP8 556 -> 474, 1039 -> 965, 1621 -> 1540; 256 experts, top-8, H 7168, I 256 at 2048 tokens bf16
// 836 -> 798, soft-FP8 770 -> 710.
//
// What bounds it: neither the matrix cores' peak nor memory.  8 experts, top-2, H 4096, I 14336, bf16, 2048 tokens: gate/up 962
// GFLOP in about 800 us (1.2 PFLOP/s), down 481 GFLOP in 465 us (1.03), where the same loop reaches 1.46 PFLOP/s on a dense 8192 x
// 8192 product of 4096 tokens; the layer 1529 -> 1335 us with the 16 x 16 products and whole-line tokens of mlk_panel8.cuh.  Counted: 6 to 8 % of the products are
// columns that pad a task; the matrix cores are busy 67 % (down: 52 %) of the cycles, at a clock that power holds at 1.87 (2.0) GHz; a CU holds
// waves 93 % (82 %: 2.5 rounds of long items) of the time, and a workgroup's first slabs and its epilogue have nothing
// beside them on the CU.  fp32 partial products of the down projection are 4 H bytes per
// routed pair and slice, written and read once (the sum over them: 26 us).
#pragma once

#include <math.h>

#include "mlk_moe_args.cuh"
#include "mlk_panel8_small.cuh"

namespace mlk {

constexpr int kWideOutPitch = 272;                             // gate/up turn-around buffer: bytes per token (128 columns)
constexpr int kWideDownPitch = 144;                            // down: bytes per token (32 fp32 rows of one wave)
constexpr size_t kWideDownOut = (size_t)8 * 128 * kWideDownPitch;

// The line of n items is cut into eight equal runs, one per XCD (workgroup id modulo 8).  Without queues every item has a workgroup of
// its own.  With them (wide_queue_pays) a workgroup per CU starts with item id / 8 of its run and goes on: queue[x] counts the items
// that have been taken from run x since, and where a run has ended its CUs help the run that has most left.
__device__ __forceinline__ int wide_item(int id, int n) {
    const int per = (n + 7) >> 3;
    const int j = id >> 3;
    return j < per ? (id & 7) * per + j : n;
}
__device__ __forceinline__ int wide_run(int n, int x) {
    const int per = (n + 7) >> 3;
    return max(0, min(per, n - x * per));
}
__device__ __forceinline__ int wide_ticket(int32_t *queue, int x, int lane) {
    int got = 0;
    if (lane == 0) got = __hip_atomic_fetch_add(queue + x * kWideQueueStep, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return got + ((int)(gridDim.x + 7 - x) >> 3);
}
// One wave: the item of a ticket of run x (valid in lane 0), or, when that run has ended, the next one of the run that has most
// left; -1 when all have ended.  A ticket that comes too late leaves its run ended for good, so there are eight attempts at most.
__device__ __forceinline__ int wide_next(int32_t *queue, int n, int x, int ticket, int lane) {
    for (;;) {
        ticket = __builtin_amdgcn_readfirstlane(ticket);
        if (ticket < wide_run(n, x)) return x * ((n + 7) >> 3) + ticket;
        int best = 0;
        if (lane < 8) {
            const int taken = __hip_atomic_load(queue + lane * kWideQueueStep, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) +
                              ((int)(gridDim.x + 7 - lane) >> 3);
            const int left = wide_run(n, lane) - taken;
            if (left > 0) best = left * 8 + lane;
        }
#pragma unroll
        for (int off = 4; off > 0; off >>= 1) best = max(best, __shfl_xor(best, off));
        best = __builtin_amdgcn_readfirstlane(best);
        if (best == 0) return -1;
        x = best & 7;
        ticket = wide_ticket(queue, x, lane);
    }
}
// The kernel's arguments (MoeArgs come first) and the place in the workgroup, taken afresh for every item: what the compiler works out
// from them in front of the loop over items is spilled there (soft-FP8 gate/up: 17 vector registers).  A kernel that calls this takes
// MoeArgs as its first argument: first_is_moe_args() is asserted where it is launched.
template <class... Rest>
constexpr bool first_is_moe_args(void (*)(MoeArgs, Rest...)) { return true; }
constexpr bool first_is_moe_args(...) { return false; }
__device__ __forceinline__ const MoeArgs &wide_args(int &lane, int &wave) {
    auto at = __builtin_amdgcn_kernarg_segment_ptr();
    int tid = threadIdx.x;
    asm volatile("" : "+s"(at), "+v"(tid));
    lane = tid & 63;
    wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    return *(const MoeArgs *)at;
}

template <class T, bool FP8, bool QUEUE, int TB>
__device__ __forceinline__ int moe_gate_up_wide(const MoeArgs &p, const MoeTask &tk, int rt, int wave, int lane) {
    extern __shared__ u32x4 win[];
    constexpr int WB = FP8 ? 1 : 2;
    using Loop = typename Panel8<T, FP8, TB, 2>::Loop;
    const int wr = wave & 3, wt = wave >> 2;
    const int groups_i = p.I >> 4;
    const uint32_t tile_row = (uint32_t)p.H * 16u * WB;          // bytes of a row group
    P8Src src;
    src.a = p.W1 + (size_t)tk.expert * 2 * p.I * p.H * WB + (size_t)rt * 8 * tile_row;
    src.b = p.X;
    // tiles 2 pair, 2 pair + 1 of the panel: quarter pair / 2, its gate tiles (even pairs) or up tiles (odd pairs)
    const int pair = FP8 ? Loop::pair(wave) : Loop::tile(wave, 0) >> 1;
    const int half = pair & 1, rg = (pair >> 1) * 2;
    const uint32_t tile0 = (uint32_t)(half * groups_i + rg) * tile_row;
    // block scales: of the half that the wave multiplies, or of the gate rows and the up rows
    constexpr int NS = Panel8<T, FP8, TB, 2>::SMALL ? 1 : 2;
    ScaleRow srow[NS];
    if constexpr (FP8) {
        src.a_off[0] = tile0 + (lane >> 5 ? tile_row : 0u) + (lane & 31) * 16;
        const int cols = p.H >> 7;
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            const int block = ((NS == 2 ? i : half) * groups_i + rt * 8) >> 3;
            srow[i] = load_scale_row(p.S1 ? p.S1 + ((size_t)tk.expert * (2 * p.I >> 7) + block) * cols : nullptr, cols, lane);
        }
    } else {
        src.a_off[0] = tile0;
        src.a_off[1] = tile0 + tile_row;
    }
    const int slots = tk.nblocks * 16;
    const int32_t *sorted = p.sorted + tk.block0 * 16;
    p8_token_rows<Loop>(src, (uint32_t)p.H * 2u, wave, lane, [&](int slot) {
        // slots without a routed pair read token 0: their columns of the product are never used
        const int id = slot < slots ? sorted[slot] : p.n_pairs;
        return id < p.n_pairs ? id / p.K : 0;
    });
    typename Loop::Acc acc;
    Loop::run(acc, src, srow, 0, p.H >> 5, wave, lane);
    __syncthreads();
    const int ticket = QUEUE && wave == 0 ? wide_ticket(p.queues, blockIdx.x & 7, lane) : 0;      // of the next item

    // the first half of the wave's rows: gate, the second: up, of its 32 columns
    uint8_t *out = reinterpret_cast<uint8_t *>(win);
    acc.each_half(lane, [&](int col, int token, f32x4 gate, f32x4 up) {
        float h[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = silu_mul(gate[e], up[e]);
        u32x2 o;
        o[0] = T::from_f32x2(h[0], h[1]);
        o[1] = T::from_f32x2(h[2], h[3]);
        *reinterpret_cast<u32x2 *>(out + (wt * TB * 32 + token) * kWideOutPitch + wr * 64 + col * 2) = o;
    });
    __syncthreads();
    // sixteen lanes store the 256 bytes of a slot; slots without a routed pair are stored too (nobody reads them)
    const int tid = wave * 64 + lane, q = tid & 15;
    uint16_t *dst = p.Hbuf + (size_t)tk.block0 * 16 * p.I + rt * 128 + q * 8;
#pragma unroll
    for (int it = 0; it < 2 * TB; ++it) {
        const int slot = it * 32 + (tid >> 4);
        if (slot < slots)
            *reinterpret_cast<u32x4 *>(dst + (size_t)slot * p.I) = *reinterpret_cast<const u32x4 *>(out + slot * kWideOutPitch + q * 16);
    }
    return ticket;
}

template <class T, bool FP8, bool QUEUE>
__device__ __forceinline__ int moe_gate_up_wide_item(const MoeArgs &p, int row_tiles, int item, int wave, int lane) {
    const MoeTask t0 = p.tasks[item / row_tiles];                // some task of the item's expert
    const int local = item - (int)t0.first * row_tiles;
    const int rt = local / t0.count;
    const MoeTask tk = p.tasks[t0.first + local % t0.count];
    switch ((tk.nblocks + 3) >> 2) {
        case 1: return moe_gate_up_wide<T, FP8, QUEUE, 1>(p, tk, rt, wave, lane);
        case 2: return moe_gate_up_wide<T, FP8, QUEUE, 2>(p, tk, rt, wave, lane);
        case 3: return moe_gate_up_wide<T, FP8, QUEUE, 3>(p, tk, rt, wave, lane);
        default: return moe_gate_up_wide<T, FP8, QUEUE, 4>(p, tk, rt, wave, lane);
    }
}

template <class T, bool FP8>
__global__ void __launch_bounds__(512) moe_gate_up_wide_kernel(MoeArgs p) {
    const int row_tiles = p.I >> 7, n_items = row_tiles * p.n_tasks[0];
    const int item = wide_item(blockIdx.x, n_items);
    if (item >= n_items) return;
    moe_gate_up_wide_item<T, FP8, false>(p, row_tiles, item, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), threadIdx.x & 63);
}

template <class T, bool FP8>
__global__ void __launch_bounds__(512) moe_gate_up_queue_kernel(MoeArgs) {
    __shared__ int s_item;
    int ticket = blockIdx.x >> 3;
    for (;;) {
        int lane, wave;
        const MoeArgs &p = wide_args(lane, wave);
        const int row_tiles = p.I >> 7, n_items = row_tiles * p.n_tasks[0];
        if (wave == 0) s_item = wide_next(p.queues, n_items, blockIdx.x & 7, ticket, lane);
        __syncthreads();                                         // also: LDS is free again
        const int item = __builtin_amdgcn_readfirstlane(s_item);
        if (item < 0) return;
        ticket = moe_gate_up_wide_item<T, FP8, true>(p, row_tiles, item, wave, lane);
    }
}

template <class T, bool FP8, bool QUEUE, int TB>
__device__ __forceinline__ int moe_down_wide(const MoeArgs &p, float *__restrict__ O, int skd, const MoeTask &tk, int rt, int sk,
                                             int wave, int lane) {
    extern __shared__ u32x4 win[];
    constexpr int WB = FP8 ? 1 : 2;
    using Loop = typename Panel8<T, FP8, TB, 2>::Loop;
    const int wr = wave & 3, wt = wave >> 2;
    const uint32_t tile_row = (uint32_t)p.I * 16u * WB;
    const int groups = p.H >> 4, rgp = rt * 16;
    P8Src src;
    src.a = p.W2 + (size_t)tk.expert * p.H * p.I * WB + (size_t)rgp * tile_row;
    src.b = p.Hbuf + (size_t)tk.block0 * 16 * p.I;
    // rows past H: a copy of the last row group, never stored
    const int tile = FP8 ? 2 * Loop::pair(wave) : Loop::tile(wave, 0);
    const int rga = min(rgp + tile, groups - 1), rgb = min(rgp + tile + 1, groups - 1);
    ScaleRow srow[1];
    if constexpr (FP8) {
        src.a_off[0] = (uint32_t)((lane >> 5 ? rgb : rga) - rgp) * tile_row + (lane & 31) * 16;
        const int cols = p.I >> 7;
        const int rgs = min(rgp + Loop::scale_tile(wave), groups - 1);
        srow[0] = load_scale_row(p.S2 ? p.S2 + ((size_t)tk.expert * (p.H >> 7) + (rgs >> 3)) * cols : nullptr, cols, lane);
    } else {
        src.a_off[0] = (uint32_t)(rga - rgp) * tile_row;
        src.a_off[1] = (uint32_t)(rgb - rgp) * tile_row;
    }
    const int slots = tk.nblocks * 16;
    p8_token_rows<Loop>(src, (uint32_t)p.I * 2u, wave, lane, [&](int slot) { return slot < slots ? slot : 0; });
    const int nwin = p.I >> 7;                                     // K slices are cut at multiples of 128 k
    const int wbeg = (int)((long long)sk * nwin / skd), wend = (int)((long long)(sk + 1) * nwin / skd);
    typename Loop::Acc acc;
    Loop::run(acc, src, srow, 4 * wbeg, 4 * (wend - wbeg), wave, lane);
    __syncthreads();
    const int ticket = QUEUE && wave == 0 ? wide_ticket(p.queues + 8 * kWideQueueStep, blockIdx.x & 7, lane) : 0;  // of the next item

    // every wave turns its 32 rows x 32 TB tokens around in its own part of LDS, one row pair after the other, and stores
    // 128 bytes of a routed pair with eight lanes
    uint8_t *out = reinterpret_cast<uint8_t *>(win) + (size_t)wave * 128 * kWideDownPitch;
    const int t8 = lane >> 3, q = lane & 7;
    const int n0 = (rgp + wr * 4) * 16;
    if (n0 >= p.H) return ticket;
    const int32_t *sorted = p.sorted + tk.block0 * 16;
#pragma unroll
    for (int pr = 0; pr < 2; ++pr) {
        acc.each(lane, [](int) {}, [&](int row, int token, f32x4 v) {
            if (row >> 5 == pr) *reinterpret_cast<f32x4 *>(out + token * kWideDownPitch + (row & 31) * 4) = v;
        });
        wave_lds_sync();
#pragma unroll 4
        for (int it = 0; it < 4 * TB; ++it) {
            const int slot = wt * TB * 32 + it * 8 + t8;
            const int id = slot < slots ? sorted[slot] : p.n_pairs;
            if (id < p.n_pairs) {
                f32x4 v = *reinterpret_cast<const f32x4 *>(out + (it * 8 + t8) * kWideDownPitch + q * 16);
                v *= T::to_f32(p.wts[id]);
                *reinterpret_cast<f32x4 *>(O + ((size_t)id * skd + sk) * p.H + n0 + pr * 32 + q * 4) = v;
            }
        }
        wave_lds_sync();
    }
    return ticket;
}

template <class T, bool FP8, bool QUEUE>
__device__ __forceinline__ int moe_down_wide_item(const MoeArgs &p, float *__restrict__ O, int skd, int row_tiles, int item, int wave,
                                                  int lane) {
    const int per_task = row_tiles * skd;
    const MoeTask t0 = p.tasks[item / per_task];
    const int local = item - (int)t0.first * per_task;
    const int rs = local / t0.count;                               // slice-major: co-running workgroups share a K window
    const int sk = rs / row_tiles, rt = rs - sk * row_tiles;
    const MoeTask tk = p.tasks[t0.first + local % t0.count];
    switch ((tk.nblocks + 3) >> 2) {
        case 1: return moe_down_wide<T, FP8, QUEUE, 1>(p, O, skd, tk, rt, sk, wave, lane);
        case 2: return moe_down_wide<T, FP8, QUEUE, 2>(p, O, skd, tk, rt, sk, wave, lane);
        case 3: return moe_down_wide<T, FP8, QUEUE, 3>(p, O, skd, tk, rt, sk, wave, lane);
        default: return moe_down_wide<T, FP8, QUEUE, 4>(p, O, skd, tk, rt, sk, wave, lane);
    }
}

template <class T, bool FP8>
__global__ void __launch_bounds__(512) moe_down_wide_kernel(MoeArgs p, float *__restrict__ O, int skd) {
    const int row_tiles = (p.H + 255) >> 8, n_items = row_tiles * skd * p.n_tasks[0];
    const int item = wide_item(blockIdx.x, n_items);
    if (item >= n_items) return;
    moe_down_wide_item<T, FP8, false>(p, O, skd, row_tiles, item, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), threadIdx.x & 63);
}

template <class T, bool FP8>
__global__ void __launch_bounds__(512) moe_down_queue_kernel(MoeArgs, float *__restrict__ O, int skd) {
    __shared__ int s_item;
    int ticket = blockIdx.x >> 3;
    for (;;) {
        int lane, wave;
        const MoeArgs &p = wide_args(lane, wave);
        const int row_tiles = (p.H + 255) >> 8, n_items = row_tiles * skd * p.n_tasks[0];
        if (wave == 0) s_item = wide_next(p.queues + 8 * kWideQueueStep, n_items, blockIdx.x & 7, ticket, lane);
        __syncthreads();                                           // also: LDS is free again
        const int item = __builtin_amdgcn_readfirstlane(s_item);
        if (item < 0) return;
        ticket = moe_down_wide_item<T, FP8, true>(p, O, skd, row_tiles, item, wave, lane);
    }
}

// Do at most n items of `slabs` k32 slabs each go through the queues?  They cost about 2 us a kernel (a ticket behind every item, a
// look at all runs at the end: with queues everywhere layers of 64 and 128 experts of H 2048 lost 1 to 3 %, at 120 to 300 us) and win
// where the XCDs' equal runs are unequal work, which takes panels of unequal widths: experts
// whose loads, three standard deviations of an even routing either way, do not all need the same columns; and enough
// rounds of long enough items to share out.
static inline bool wide_queue_pays(const MoeArgs &a, int n, int slabs) {
    const double mean = (double)a.n_pairs / a.E, spread = 3 * sqrt(mean);
    if (ceil(fmax(mean - spread, 1) / 64) == ceil((mean + spread) / 64)) return false;
    return n > device_cus() && (double)n / device_cus() * (slabs + 8) >= 350;
}

template <class T, bool FP8>
int launch_moe_wide(const MoeArgs &a, int max_tasks, float *obuf, int skd, hipStream_t s) {
    constexpr size_t ring = p8_ring_bytes<FP8, 2, 4>();
    constexpr size_t lds_up = ring, lds_down = ring > kWideDownOut ? ring : kWideDownOut;
    static bool ready_up[2][64] = {}, ready_down[2][64] = {};
    const int items_up = (a.I >> 7) * max_tasks, items_down = ((a.H + 255) >> 8) * skd * max_tasks;
    const bool queue_up = wide_queue_pays(a, items_up, a.H >> 5), queue_down = wide_queue_pays(a, items_down, (a.I >> 5) / skd);
    static_assert(first_is_moe_args(moe_gate_up_queue_kernel<T, FP8>) && first_is_moe_args(moe_down_queue_kernel<T, FP8>),
                  "wide_args() reads MoeArgs where the kernel's arguments begin");
    const auto up = queue_up ? &moe_gate_up_queue_kernel<T, FP8> : &moe_gate_up_wide_kernel<T, FP8>;
    const auto down = queue_down ? &moe_down_queue_kernel<T, FP8> : &moe_down_wide_kernel<T, FP8>;
    int rc = panel_lds_attribute(up, lds_up, ready_up[queue_up]);
    if (rc != MLK_OK) return rc;
    rc = panel_lds_attribute(down, lds_down, ready_down[queue_down]);
    if (rc != MLK_OK) return rc;
    up<<<queue_up ? device_cus() : (items_up + 7) / 8 * 8, 512, lds_up, s>>>(a);
    MLK_LAUNCH_CHECK();
    down<<<queue_down ? device_cus() : (items_down + 7) / 8 * 8, 512, lds_down, s>>>(a, obuf, skd);
    MLK_LAUNCH_CHECK();
    return MLK_OK;
}

}  // namespace mlk
