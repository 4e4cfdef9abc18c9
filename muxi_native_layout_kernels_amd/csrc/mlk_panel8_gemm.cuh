// The eight-wave panel GeMM (main loops: mlk_panel8.cuh, mlk_panel8_small.cuh) and what it shares with the other panel kernels: arguments, fold.
#pragma once

#include "mlk_panel8_small.cuh"

namespace mlk {

struct PanelArgs {
    const uint8_t *A;
    const uint16_t *B;
    uint16_t *C;
    const uint16_t *bias;
    const float *scale;
    f32x4 *partial;      // [SK][sliced tiles][4 waves][quads of a wave][two planes of 64 x 8 bytes]
    int *counters;       // [sliced tiles], zero between calls
    int M, N, K;
    int SK;              // K slices of the row tiles from whole_groups * 8 on
    int whole_groups;    // groups of eight row tiles in front that are not sliced (0: every row tile has SK slices)
    int row_tiles, token_tiles;
    float alpha;
};

// Arguments of the eight-wave panels (gemm_panel8_kernel, gemm_panel8_fold_kernel), panels of 128 pr rows x 64 tb tokens.
//
// The panels form one line (band 0), or one line per XCD (band > 0).  The first `whole` panels of a line are
// computed by one workgroup each; the k windows (64 k) of those that follow are dealt to `deal` workgroups in equal
// contiguous runs, whatever panel they belong to.  A run that covers part of a panel leaves its fp32 sums in a slot of its own
// (the first slot of its workgroup: the panel its run starts in; the second: the one it ends in), and gemm_panel8_fold_kernel adds
// the slots of a panel in the order of k and stores the result.
struct Panel8Args {
    const uint8_t *A;
    const uint16_t *B;
    uint16_t *C;
    const uint16_t *bias;
    const float *scale;
    f32x4 *partial;      // [line][deal][slots] of slots of 128 pr rows x cols tokens (p8_slot_quad)
    int M, N, K;
    int row_tiles, token_tiles;
    int cols;            // tokens of a slot: 64 tb, or the call's tokens in blocks of 16 where one token tile holds them all (32 to 48
                         // tokens in slices are then no larger than the narrow kernels' partial sums)
    bool rows_first;     // one line: the row tiles of a token tile are neighbours, else the token tiles of a row tile
    int band, chunk;     // groups of eight row tiles and token tiles that neighbouring workgroups of an XCD cover
    int panels;          // of the longest line
    int whole, deal;     // of one line
    int slots;           // per dealt workgroup: 1 where no run crosses from one panel into the next, else 2
    int b_native, c_native;  // activations in layout B, output in layout C (else row-major)
    float alpha;
};

// Panel u of a line; false when there is none.
__device__ __forceinline__ bool p8_panel(const Panel8Args &p, int line, int u, int &rt, int &tt) {
    if (p.band > 0) {
        const int TT = p.token_tiles, groups8 = (p.row_tiles + 7) >> 3, RB = p.band, TC = p.chunk;
        const int band = u / (RB * TT);
        const int nb = min(RB, groups8 - band * RB);           // groups of row tiles in this band
        const int v = u - band * RB * TT;
        const int c = v / (nb * TC);
        const int tc = min(TC, TT - c * TC);                   // token tiles in this chunk
        const int w = v - c * nb * TC;
        tt = c * TC + w % tc;
        rt = (band * RB + w / tc) * 8 + line;
        return rt < p.row_tiles;
    }
    const int inner = p.rows_first ? p.row_tiles : p.token_tiles, a = u / inner, b = u - a * inner;
    rt = p.rows_first ? b : a;
    tt = p.rows_first ? a : b;
    return rt < p.row_tiles;
}

// Where the four sums of rows 4 quad .. + 3 (quad < 8) of row pair `pair` of the panel and token block + t lie in
// a panel's sums of `cols` tokens.  A block of 32 tokens is one run per row pair; the last block may have 16 tokens.
__device__ __forceinline__ int p8_slot_quad(int cols, int pair, int block, int width, int quad, int t) {
    return (pair * cols + block) * 8 + quad * width + t;
}

// Element offset of 8 rows n .. n + 7 (n % 8 == 0) of token tok in a layout-C output of m tokens.
__device__ __forceinline__ size_t native_c_offset(int n, int tok, int m) {
    return (((size_t)(n >> 5) * (m >> 4) + (tok >> 4)) * 4 + ((n >> 3) & 3)) * 128 + (tok & 15) * 8;
}

// What happens to the accumulators of a panel: scaled and stored, or (K slices) handed over as fp32 partials that the
// last workgroup to arrive adds in slice order.  acc[pr][tb] covers the row groups rg0 + 2 pr, + 1 and the 32 tokens from
// tok0 + 32 tb on; kTileWaves waves per workgroup, each with PR x TB accumulators; the fold fetches FB accumulators at a time.
template <class T, int PR, int TB, int FB>
__device__ __forceinline__ void panel_finish(const PanelArgs &p, f32x16 (&acc)[PR][TB], int rg0, int tok0, int SK, int sk,
                                             int rt, int tt, int wave, int lane, int *s_last) {
    const int groups = p.N >> 4;
    // accumulator element 4 g + e of lane 32 h + c: weight row 8 g + 4 h + e of the pair's 32, token c of the block's 32
    const int half = lane >> 5, c32 = lane & 31;
    auto epilogue = [&](int pr, int tb, int g, f32x4 v) {
        const int n = (rg0 + 2 * pr) * 16 + 8 * g + 4 * half;
        const int tok = tok0 + tb * 32 + c32;
        if ((n >> 4) >= groups || tok >= p.M) return;
        float o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            o[i] = p.alpha * v[i];
            if (p.bias) o[i] += T::to_f32(p.bias[n + i]);
        }
        store4<T>(p.C + (size_t)tok * p.N + n, o[0], o[1], o[2], o[3]);
    };
    auto quad = [&](const f32x16 &v, int g) { return f32x4{v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]}; };
    if (SK == 1) {
#pragma unroll
        for (int pr = 0; pr < PR; ++pr)
#pragma unroll
            for (int tb = 0; tb < TB; ++tb)
#pragma unroll
                for (int g = 0; g < 4; ++g) epilogue(pr, tb, g, quad(acc[pr][tb], g));
        return;
    }
    const int tile = (rt - p.whole_groups * 8) * p.token_tiles + tt;               // among the sliced tiles
    const int tiles = (p.row_tiles - p.whole_groups * 8) * p.token_tiles;
    // 64-lane group of quad jj of this wave in slice s (two planes of 8-byte halves, see st_agent_planar)
    auto group_at = [&](int s, int jj) -> f32x4 * {
        return p.partial + ((((size_t)s * tiles + tile) * kTileWaves + wave) * (PR * TB * 4) + jj) * 64;
    };
    // partials travel as agent-scope (write-through / always-miss) accesses, like in the narrow kernels; a release /
    // acquire fence pair around ordinary stores was measured slower (it writes back and invalidates a whole L2)
#pragma unroll
    for (int pr = 0; pr < PR; ++pr)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
            for (int g = 0; g < 4; ++g) st_agent_planar(group_at(sk, (pr * TB + tb) * 4 + g), 64, lane, quad(acc[pr][tb], g));
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0) {
        int prev = __hip_atomic_fetch_add(&p.counters[tile], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *s_last = (prev == SK - 1);
        if (*s_last) __hip_atomic_store(&p.counters[tile], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!*s_last) return;
    // slice order; the loads of the next slice are in flight while the current one is added (a round trip to
    // memory per slice would otherwise be paid in full: these loads bypass the caches).  FB accumulators are fetched,
    // added and stored at a time, in registers of their own: the published accumulators are dead, and summing into them would
    // keep all of them alive to the end.
    static_assert(TB % FB == 0, "fetch groups are whole accumulators of one row pair");
#pragma unroll
    for (int pr = 0; pr < PR; ++pr) {
#pragma unroll
        for (int t0b = 0; t0b < TB; t0b += FB) {
            f32x16 sum[FB];
#pragma unroll
            for (int tb = 0; tb < FB; ++tb)
#pragma unroll
                for (int e = 0; e < 16; ++e) sum[tb][e] = 0.f;
            f32x4 t0[FB * 4], t1[FB * 4];
            auto fetch = [&](f32x4 (&t)[FB * 4], int sl) {
#pragma unroll
                for (int jj = 0; jj < FB * 4; ++jj) t[jj] = ld_agent_planar(group_at(sl, (pr * TB + t0b) * 4 + jj), 64, lane);
            };
            auto add = [&](const f32x4 (&t)[FB * 4]) {
#pragma unroll
                for (int tb = 0; tb < FB; ++tb)
#pragma unroll
                    for (int e = 0; e < 16; ++e) sum[tb][e] += t[tb * 4 + (e >> 2)][e & 3];
            };
            fetch(t0, 0);
            for (int sl = 0; sl < SK; sl += 2) {
                if (sl + 1 < SK) fetch(t1, sl + 1);
                add(t0);
                if (sl + 1 < SK) {
                    if (sl + 2 < SK) fetch(t0, sl + 2);
                    add(t1);
                }
            }
#pragma unroll
            for (int tb = 0; tb < FB; ++tb)
#pragma unroll
                for (int g = 0; g < 4; ++g) epilogue(pr, t0b + tb, g, quad(sum[tb], g));
        }
    }
}

// Output of an eight-wave panel that is computed whole: every wave turns its 32 PR rows x 32 TB tokens around in LDS (the
// ring is free by then; 16 bytes more per token than its rows take, so that the 8-byte pieces of 32 tokens meet each bank at
// most twice).  Row-major output: whole 128-byte lines (PR = 2) or halves of them that two neighbouring waves complete, eight
// or sixteen tokens per instruction.  Stored straight from the accumulators, a lane's four rows of one
// token are 8 bytes in a line that fifteen other instructions complete: 67 MB of output took 23 us that way.
// Layout C: 32 rows of 16 tokens are one run of 1 KiB, a store each.
__host__ __device__ constexpr int p8_out_pitch(int pr) { return 64 * pr + 16; }      // bytes per token in the turn-around buffer
template <bool FP8, int PR, int TB>
constexpr size_t p8_lds_bytes() {
    const size_t ring = p8_ring_bytes<FP8, PR, TB>(), out = (size_t)8 * 32 * TB * p8_out_pitch(PR);
    return ring > out ? ring : out;
}
template <class T, int PR, int TB, class Acc>
__device__ __forceinline__ void p8_store_panel(const Panel8Args &p, const Acc &acc, int rg0, int tok0, int wave, int lane,
                                               u32x4 *win) {
    constexpr int PITCH = p8_out_pitch(PR);
    uint8_t *buf = reinterpret_cast<uint8_t *>(win) + (size_t)wave * 32 * TB * PITCH;
    const int n0 = rg0 * 16;                                   // first of the wave's 32 PR rows
    auto put = [&](int row, int token, f32x4 v, const float (&bias)[4]) {
        u32x2 o;
        o[0] = T::from_f32x2(p.alpha * v[0] + bias[0], p.alpha * v[1] + bias[1]);
        o[1] = T::from_f32x2(p.alpha * v[2] + bias[2], p.alpha * v[3] + bias[3]);
        *reinterpret_cast<u32x2 *>(buf + token * PITCH + row * 2) = o;
    };
    // Asked once whether there is a bias: a branch for every four rows and token block, each over code that is fetched for the first time,
    // took 0.2 us of a call
    float bias[4] = {0.f, 0.f, 0.f, 0.f};
    if (p.bias == nullptr) {
        acc.each(lane, [](int) {}, [&](int row, int token, f32x4 v) { put(row, token, v, bias); });
    } else {
        auto rows = [&](int row) {
#pragma unroll
            for (int e = 0; e < 4; ++e) bias[e] = n0 + row < p.N ? T::to_f32(p.bias[n0 + row + e]) : 0.f;
        };
        acc.each(lane, rows, [&](int row, int token, f32x4 v) { put(row, token, v, bias); });
    }
    if (p.c_native) {
        // lane 16 q + t: octet q of token t of each block of 16 tokens x 32 rows
        const int t16 = lane & 15, q = lane >> 4;
#pragma unroll
        for (int pr = 0; pr < PR; ++pr)
#pragma unroll
            for (int it = 0; it < 2 * TB; ++it) {
                const int tok = tok0 + it * 16 + t16, n = n0 + pr * 32 + q * 8;
                const u32x4 v = *reinterpret_cast<const u32x4 *>(buf + (it * 16 + t16) * PITCH + pr * 64 + q * 16);
                if (n < p.N && tok < p.M) *reinterpret_cast<u32x4 *>(p.C + native_c_offset(n, tok, p.M)) = v;
            }
        return;
    }
    // lane 4 PR t + q: 16 bytes (8 rows) q of token t of each group of 16 / PR tokens
    constexpr int LPT = 4 * PR, TPI = 64 / LPT;
    const int t8 = lane / LPT, q = lane % LPT;
    const bool rows_ok = n0 + q * 8 < p.N;
#pragma unroll
    for (int it = 0; it < 32 * TB / TPI; ++it) {
        const int token = it * TPI + t8;
        const u32x4 v = *reinterpret_cast<const u32x4 *>(buf + token * PITCH + q * 16);
        if (rows_ok && tok0 + token < p.M) *reinterpret_cast<u32x4 *>(p.C + (size_t)(tok0 + token) * p.N + n0 + q * 8) = v;
    }
}

// ---------------------------------------------------------------------------------------------------------------
// Panels of 128 PR rows x 64 MAXTB tokens on the eight-wave loop of mlk_panel8.cuh.
//
// Order of the panels (p8_panel).  In bands, for grids of several rounds: the workgroup ids of an XCD walk
// bands of p.band groups of eight row tiles in chunks of
// p.chunk token tiles, so that the 32 workgroups an XCD runs at a time cover 8 x 4 (row tiles x token tiles) and share
// both operands through its L2; with the token tiles of two row tiles side by side (2 x 16) the same product took
// 17 % longer (8192 x 8192, 4096 tokens, 491 against 413 us; timed on a loop before this one, of 32x32x16 products on tokens in
// pieces of 64 bytes).
// In one line, token tiles fastest, for few panels: dealing whole row tiles to XCDs leaves half of them idle at 512 rows.  The
// workgroups of the line (one per panel, or those that share the k windows) are cut into eight runs, one per XCD.
template <class T, bool FP8, int PR, int TB, int MAXTB>
__device__ __forceinline__ void gemm_panel8(const Panel8Args &p, int rt, int tt, int slab0, int nslab, f32x4 *slot) {
    extern __shared__ u32x4 win[];
    constexpr int WBYTES = FP8 ? 1 : 2;
    using Loop = typename Panel8<T, FP8, TB, PR>::Loop;
    // Taken afresh for every run: what the compiler works out from it in front of the loop over runs is spilled there (soft-FP8 256 x 256:
    // 9 vector registers).  Not in soft-FP8 panels of 128 x 128 and 128 x 192, which spill nothing either way and whose loop is scheduled
    // better without (products of 12 to 50 us: 1.4 and 2.9 % faster; the other shapes are level or slower without).
    int tid = threadIdx.x;
    if constexpr (!(FP8 && PR == 1 && (MAXTB == 2 || MAXTB == 3))) asm volatile("" : "+v"(tid));
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave & 3, wt = wave >> 2;
    const int groups = p.N >> 4;
    const int rgp = rt * 8 * PR;                               // first row group of the panel
    const int rg0 = rgp + wr * 2 * PR;                         // of this wave
    const int tok0 = tt * 64 * MAXTB;

    // sources of this wave's loads: its weight tiles of the panel (rows past N: a copy of the last row
    // group, never stored), its token chunks (tokens past M: the last token)
    P8Src src;
    src.a = p.A + (size_t)rgp * p.K * 16 * WBYTES;
    src.b = p.B;
    ScaleRow srow[1];
    if constexpr (FP8) {
        const int t0 = 2 * Loop::pair(wave);
        const int rga = min(rgp + t0, groups - 1), rgb = min(rgp + t0 + 1, groups - 1);
        src.a_off[0] = (uint32_t)((lane >> 5 ? rgb : rga) - rgp) * (uint32_t)p.K * 16u + (lane & 31) * 16;
        const int scale_cols = (p.K + 127) >> 7;
        const int rgs = min(rgp + Loop::scale_tile(wave), groups - 1);
        srow[0] = load_scale_row(p.scale ? p.scale + (size_t)(rgs >> 3) * scale_cols : nullptr, scale_cols, lane);
    } else {
#pragma unroll
        for (int i = 0; i < PR; ++i)
            src.a_off[i] = (uint32_t)(min(rgp + Loop::tile(wave, i), groups - 1) - rgp) * (uint32_t)p.K * 32u;
    }
    auto token_of = [&](int slot) { return min(tok0 + slot, p.M - 1); };
    if (p.b_native) p8_token_native<Loop>(src, p.M, wave, lane, token_of);
    else p8_token_rows<Loop>(src, (uint32_t)p.K * 2u, wave, lane, token_of);
    typename Loop::Acc acc;
    Loop::run(acc, src, srow, slab0, nslab, wave, lane);
    if (slot == nullptr) {
        __syncthreads();
        p8_store_panel<T, PR, TB>(p, acc, rg0, tok0 + wt * 32 * TB, wave, lane, win);
        return;
    }
    const int cols = min(p.cols, 64 * TB);
    acc.each(lane, [](int) {}, [&](int row, int token, f32x4 v) {
        const int block = (wt * TB + (token >> 5)) * 32, width = min(32, cols - block);
        if ((token & 31) < width) slot[p8_slot_quad(cols, wr * PR + (row >> 5), block, width, (row & 31) >> 2, token & 31)] = v;
    });
}

// Token columns / 64 that token tile tt multiplies: the last tile those that cover it (28672 x 4096 bf16 at 700 tokens 196 ->
// 193 us, 13824 x 5120 at 3000 tokens 372 -> 367 us).
__device__ __forceinline__ int p8_columns(int m, int tt, int maxtb) { return min(maxtb, (m - tt * 64 * maxtb + 63) >> 6); }

template <class T, bool FP8, int PR, int MAXTB>
__global__ void __launch_bounds__(512) gemm_panel8_kernel(Panel8Args p) {
    int line = blockIdx.x & 7, u = blockIdx.x >> 3;
    if (p.band == 0) {
        const int n = p.whole + p.deal, run = (n + 7) >> 3;        // one of the two is zero
        if (u >= run) return;
        u += line * run;
        line = 0;
    }
    const int windows = p.K >> 6;
    int at = u * windows, end = at + windows;                      // in k windows of the line
    const int j = u - p.whole;
    if (j >= 0) {
        if (j >= p.deal) return;
        const int total = (p.panels - p.whole) * windows;
        at = p.whole * windows + (int)((long long)j * total / p.deal);
        end = p.whole * windows + (int)((long long)(j + 1) * total / p.deal);
    }
    for (int seg = 0; at < end; seg = 1) {
        const int panel = at / windows, w0 = at - panel * windows, n = min(windows - w0, end - at);
        int rt, tt;
        if (p8_panel(p, line, panel, rt, tt)) {
            f32x4 *slot = n == windows ? nullptr : p.partial + ((size_t)(line * p.deal + j) * p.slots + seg) * (32 * PR * p.cols);
            const int tb = p8_columns(p.M, tt, MAXTB);
            if (MAXTB == 1 || tb == 1) gemm_panel8<T, FP8, PR, 1, MAXTB>(p, rt, tt, 2 * w0, 2 * n, slot);
            if constexpr (MAXTB >= 2)
                if (tb == 2) gemm_panel8<T, FP8, PR, 2, MAXTB>(p, rt, tt, 2 * w0, 2 * n, slot);
            if constexpr (MAXTB >= 3)
                if (tb == 3) gemm_panel8<T, FP8, PR, 3, MAXTB>(p, rt, tt, 2 * w0, 2 * n, slot);
            if constexpr (MAXTB >= 4)
                if (tb == 4) gemm_panel8<T, FP8, PR, 4, MAXTB>(p, rt, tt, 2 * w0, 2 * n, slot);
        }
        at += n;
        __syncthreads();                                       // the next panel's first slabs go where this one's output was turned
    }
}

// Adds the slots of the panels whose k windows were dealt to several workgroups, in the order of k, and stores them.  One wave per
// 32 rows x 32 tokens and half of the rows' groups of eight; grid (waves of a panel / 4, panels of a line that are dealt, lines).
// A second launch: added by the last workgroup of a panel to arrive instead, the fold took 8 us for eight slices of a 128 x 64
// panel and 21 us for two of a 256 x 256 one (one CU reads all of it behind three round trips to memory).
template <class T>
__global__ void __launch_bounds__(256) gemm_panel8_fold_kernel(Panel8Args p, int pr_n, int maxtb) {
    const int line = blockIdx.z, local = blockIdx.y;
    int rt, tt;
    if (!p8_panel(p, line, p.whole + local, rt, tt)) return;
    const int tb_n = p8_columns(p.M, tt, maxtb);
    const int lane = threadIdx.x & 63;
    int i = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);      // (wave, row pair, token block, half)
    if (i >= 16 * pr_n * tb_n) return;
    const int gp = (i & 1) * 2;
    i >>= 1;
    const int tb = i % tb_n, pr = i / tb_n % pr_n, wave = i / (tb_n * pr_n);
    const int cols = min(p.cols, 64 * tb_n), block = ((wave >> 2) * tb_n + tb) * 32, width = min(32, cols - block);     // of the panel's tokens
    if ((lane & 31) >= width) return;

    const int windows = p.K >> 6, total = (p.panels - p.whole) * windows, first = local * windows;
    auto owner = [&](int at) { return (int)((((long long)at + 1) * p.deal - 1) / total); };
    const int j0 = owner(first), j1 = owner(first + windows - 1);
    if (j0 == j1) return;                                      // one workgroup computed and stored it
    const bool j0_starts = (int)((long long)j0 * total / p.deal) == first;
    const size_t slot_quads = (size_t)32 * pr_n * p.cols;
    const int quad = p8_slot_quad(cols, (wave & 3) * pr_n + pr, block, width, 2 * gp + (lane >> 5), lane & 31);
    auto at = [&](int j) {
        return p.partial + ((size_t)(line * p.deal + j) * p.slots + (j == j0 && !j0_starts)) * slot_quads + quad;
    };
    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;
    for (int j = j0; j <= j1; j += 8) {                        // eight slots in flight: a round trip each if fetched one by one
        f32x4 t[8][2];
#pragma unroll
        for (int d = 0; d < 8; ++d)
            if (j + d <= j1) t[d][0] = at(j + d)[0], t[d][1] = at(j + d)[2 * width];
#pragma unroll
        for (int d = 0; d < 8; ++d)
            if (j + d <= j1) s0 += t[d][0], s1 += t[d][1];
    }
    // lane 32 h + c holds rows 8 gp + 4 h .. + 3 (s0) and 8 gp + 8 + 4 h .. + 3 (s1) of token c; swapped between the halves it
    // has rows 8 (gp + h) .. + 7
    float o[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(s0[e]), __float_as_uint(s1[e]), false, false);
        o[e] = __uint_as_float(x[0]);
        o[4 + e] = __uint_as_float(x[1]);
    }
    const int n = (rt * 8 * pr_n + (wave & 3) * 2 * pr_n + 2 * pr) * 16 + 8 * (gp + (lane >> 5));
    const int tok = tt * 64 * maxtb + block + (lane & 31);
    if (n >= p.N || tok >= p.M) return;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        o[e] *= p.alpha;
        if (p.bias) o[e] += T::to_f32(p.bias[n + e]);
    }
    const u32x4 v = {T::from_f32x2(o[0], o[1]), T::from_f32x2(o[2], o[3]), T::from_f32x2(o[4], o[5]), T::from_f32x2(o[6], o[7])};
    *reinterpret_cast<u32x4 *>(p.C + (p.c_native ? native_c_offset(n, tok, p.M) : (size_t)tok * p.N + n)) = v;
}

template <class T, bool FP8, int PR, int TB>
static int launch_panel8_shape(const Panel8Args &p, hipStream_t s) {
    constexpr size_t lds = p8_lds_bytes<FP8, PR, TB>();
    static bool ready_on[64] = {};
    const int rc = panel_lds_attribute(&gemm_panel8_kernel<T, FP8, PR, TB>, lds, ready_on);
    if (rc != MLK_OK) return rc;
    gemm_panel8_kernel<T, FP8, PR, TB><<<p.band > 0 ? (p.whole + p.deal) * 8 : (p.whole + p.deal + 7) / 8 * 8, 512, lds, s>>>(p);
    MLK_LAUNCH_CHECK();
    if (p.deal > 0) {
        gemm_panel8_fold_kernel<T><<<dim3(4 * PR * TB, p.panels - p.whole, p.band > 0 ? 8 : 1), 256, 0, s>>>(p, PR, TB);
        MLK_LAUNCH_CHECK();
    }
    return MLK_OK;
}

// Panels of 128 pr rows x 64 tb tokens; p's tiles, order and deal belong to that shape.
template <class T, bool FP8>
int launch_panel8(const Panel8Args &p, int pr, int tb, hipStream_t s) {
    switch (pr * 8 + tb) {
        case 8 + 1: return launch_panel8_shape<T, FP8, 1, 1>(p, s);
        case 8 + 2: return launch_panel8_shape<T, FP8, 1, 2>(p, s);
        case 8 + 3: return launch_panel8_shape<T, FP8, 1, 3>(p, s);
        case 8 + 4: return launch_panel8_shape<T, FP8, 1, 4>(p, s);
        case 16 + 1: return launch_panel8_shape<T, FP8, 2, 1>(p, s);
        case 16 + 2: return launch_panel8_shape<T, FP8, 2, 2>(p, s);
        case 16 + 3: return launch_panel8_shape<T, FP8, 2, 3>(p, s);
        case 16 + 4: return launch_panel8_shape<T, FP8, 2, 4>(p, s);
    }
    return fail(MLK_ERR_INVALID, "gemm: no such panel shape");
}

}  // namespace mlk
