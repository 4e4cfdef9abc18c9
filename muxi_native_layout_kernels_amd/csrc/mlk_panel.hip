// Kernel id 3: panel GeMM for more than 64 tokens over layout-A weights (row-major activations and
// output), where the product is bound by the matrix cores and no longer by the weight stream.
//
// A workgroup of four waves computes a panel of 256 weight rows x 128 tokens over one of SK slices
// of K with v_mfma_f32_32x32x16 (one wave per SIMD issues the 16x16x32 form at little more than half
// rate; the 32x32 form runs at nine tenths of peak from a single wave).  Every wave owns four row
// groups (two pairs of 32 rows) and all four blocks of 32 tokens: eight 32x32 accumulators.  Two other
// shapes exist: 256 rows x 256 tokens (sixteen accumulators, k windows of 64 instead of 128) when that
// makes fewer rounds of one workgroup per CU, and 128 rows x 128 tokens (one pair of row groups per
// wave) while panels are too few to give every CU one.
//
// Weights come straight from global memory, two k windows ahead in a register ring.  A layout-A
// tile (16 rows x 32 k: lane 16 q + r holds row r, k octet q) is not the 32x32x16 operand (lane
// 32 g + i holds row i, k octet g of a 16-wide k slice), but two vertically adjacent tiles X, Y become
// the two operands of their 32 k with two lane swaps per register: v_permlane16_swap turns the
// 16-lane rows [X0 X1 X2 X3], [Y0 Y1 Y2 Y3] into [X0 Y0 X2 Y2], [X1 Y1 X3 Y3], v_permlane32_swap
// then into [X0 Y0 X1 Y1] (k octets 0, 1 of rows 0..31) and [X2 Y2 X3 Y3] (octets 2, 3).
//
// The activations of a k window are fetched once per workgroup with 16-byte loads two windows ahead
// (they wait in registers) and parked in LDS one window ahead in operand order: granule
// ((t*TB + tb)*4 + octet)*33 + token (+ 4 t) for k tile t, token block tb, so that an operand is two
// runs of 32 consecutive granules for ds_read_b128 and the granules a token row contributes fall into
// different banks.  Three LDS buffers, one barrier per window; within a window the LDS reads and the
// global loads are scheduled between the MFMAs (sched_group_barrier).
//
// Grid: the token tiles of one row tile run next to each other on one XCD (workgroup id modulo 8
// picks the XCD), so the weights of a row tile are read from HBM once and served to the other token
// tiles by that XCD's L2.  K slices fold like in the row-shared kernel: fp32 partials with
// agent-scope stores, the last workgroup to arrive adds them in slice order.
#include "mlk_panel_loop.cuh"
#include "mlk_panel8.cuh"

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
    int band, chunk;     // gemm_panel8_kernel: groups of row tiles and token tiles that neighbouring workgroups of an XCD cover
    float alpha;
};

// What happens to the accumulators of a panel: scaled and stored, or (K slices) handed over as fp32 partials that the
// last workgroup to arrive adds in slice order.  acc[pr][tb] covers the row groups rg0 + 2 pr, + 1 and the 32 tokens from
// tok0 + 32 tb on; NWAVES waves per workgroup, each with PR x TB accumulators; the fold fetches FB accumulators at a time.
template <class T, int PR, int TB, int NWAVES, int FB>
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
        return p.partial + ((((size_t)s * tiles + tile) * NWAVES + wave) * (PR * TB * 4) + jj) * 64;
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
    // added and stored at a time (all of a row pair's where the registers allow it), in registers of their own: the
    // published accumulators are dead, and summing into them kept all of them alive to the end, at 256 registers and a
    // hundred spilled ones in the eight-wave kernels (now 234 and none: 4096 x 11008 at 1024 tokens in four slices, fp16 134 ->
    // 108 us, bf16 131 -> 105 us; 8192 x 8192 fp16 at 512 tokens in two 148 -> 122 us).
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

template <class T, bool FP8, int TB, int PR>
__global__ void __launch_bounds__(256, 1) gemm_panel_kernel(PanelArgs p) {
    extern __shared__ u32x4 win[];
    __shared__ int s_last;
    constexpr int R = 2 * PR, KW = panel_kw(TB);               // PR pairs of row groups per wave
    constexpr int WBYTES = FP8 ? 1 : 2;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // workgroup -> (row tile, k slice, token tile): per XCD first the groups of eight row tiles that are computed
    // whole, then the sliced ones
    const int xcd = blockIdx.x & 7;
    int u = blockIdx.x >> 3;
    const int whole_wgs = p.whole_groups * p.token_tiles;
    const bool sliced = u >= whole_wgs;
    const int SK = sliced ? p.SK : 1;
    if (sliced) u -= whole_wgs;
    const int tt = u % p.token_tiles;
    u /= p.token_tiles;
    const int sk = u % SK;
    const int rt = ((sliced ? p.whole_groups : 0) + u / SK) * 8 + xcd;
    if (rt >= p.row_tiles) return;                            // the grid is padded to whole groups of eight row tiles

    const int groups = p.N >> 4;
    const int rg0 = (rt * kTileWaves + wave) * R;
    const int tok0 = tt * (TB * 32);
    const int nwin_total = p.K / (KW * 32);
    const int wbeg = (int)((long long)sk * nwin_total / SK);
    const int nwin = (int)((long long)(sk + 1) * nwin_total / SK) - wbeg;
    const int scale_cols = (p.K + 127) >> 7;

    const uint8_t *abase[R];                                  // wave-uniform; the lane offset is added per load
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int rg = min(rg0 + r, groups - 1);              // rows past N are computed on a copy and never stored
        abase[r] = p.A + (size_t)rg * p.K * 16 * WBYTES;
    }
    ScaleRow srow;
    if (FP8) srow = load_scale_row(p.scale ? p.scale + (size_t)(min(rg0, groups - 1) >> 3) * scale_cols : nullptr, scale_cols, lane);

    // activation staging: a window is 32 TB tokens x GPR granules (k tile colg >> 2, octet colg & 3); granule i of
    // this thread is token trow + RP i of the panel, k granule colg
    constexpr int GPR = KW * 4, RP = 256 / GPR, NG = TB * 32 / RP;
    const int colg = tid % GPR, trow = tid / GPR;
    uint32_t boff[NG];
#pragma unroll
    for (int i = 0; i < NG; ++i) {
        const int tok = min(tok0 + trow + RP * i, p.M - 1);
        boff[i] = (uint32_t)tok * (uint32_t)p.K + colg * 8;
    }
    f32x16 acc[PR][TB];
#pragma unroll
    for (int pr = 0; pr < PR; ++pr)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[pr][tb][e] = 0.f;

    ScaleRow srows[PR];
#pragma unroll
    for (int pr = 0; pr < PR; ++pr) srows[pr] = srow;          // the row groups of a wave lie in one 128-row block
    PanelLoop<T, FP8, TB, PR>::run(acc, abase, srows, p.B, boff, wbeg, nwin, win);

    panel_finish<T, PR, TB, kTileWaves, TB>(p, acc, rg0, tok0, SK, sk, rt, tt, wave, lane, &s_last);
}

// 256 x 128 panels on the loop of mlk_panel_lds.cuh (four waves, LDS as the prefetch buffer; soft-FP8: two workgroups
// per CU).  Same grid and fold as gemm_panel_kernel.
template <class T, bool FP8, int RING>
__global__ void __launch_bounds__(256, 2) gemm_panel_lds_kernel(PanelArgs p) {
    extern __shared__ u32x4 win[];
    constexpr int TB = 4, PR = 2, R = 4;
    constexpr int WBYTES = FP8 ? 1 : 2;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int xcd = blockIdx.x & 7;
    int u = blockIdx.x >> 3;
    const int whole_wgs = p.whole_groups * p.token_tiles;
    const bool sliced = u >= whole_wgs;
    const int SK = sliced ? p.SK : 1;
    if (sliced) u -= whole_wgs;
    const int tt = u % p.token_tiles;
    u /= p.token_tiles;
    const int sk = u % SK;
    const int rt = ((sliced ? p.whole_groups : 0) + u / SK) * 8 + xcd;
    if (rt >= p.row_tiles) return;

    const int groups = p.N >> 4;
    const int rg0 = (rt * kTileWaves + wave) * R;
    const int tok0 = tt * (TB * 32);
    const int nwin_total = p.K / 128;                          // slices are cut in windows of 128 k, as the host counts them
    const int wbeg = (int)((long long)sk * nwin_total / SK);
    const int nwin = (int)((long long)(sk + 1) * nwin_total / SK) - wbeg;
    const int scale_cols = (p.K + 127) >> 7;
    const uint8_t *abase[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int rg = min(rg0 + r, groups - 1);              // rows past N are computed on a copy and never stored
        abase[r] = p.A + (size_t)rg * p.K * 16 * WBYTES;
    }
    ScaleRow srows[PR];
    if (FP8) {
        srows[0] = load_scale_row(p.scale ? p.scale + (size_t)(min(rg0, groups - 1) >> 3) * scale_cols : nullptr, scale_cols, lane);
        srows[1] = srows[0];                                   // the row groups of a wave lie in one 128-row block
    }
    auto row_off = [&](int slot) -> uint32_t { return (uint32_t)min(tok0 + slot, p.M - 1) * (uint32_t)p.K; };
    f32x16 acc[PR][TB];
#pragma unroll
    for (int pr = 0; pr < PR; ++pr)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[pr][tb][e] = 0.f;
    PanelLoopLds<T, FP8, TB, RING>::run(acc, abase, srows, p.B, row_off, 4 * wbeg, 4 * nwin, win);
    __syncthreads();                                           // the ring is given up: its first word takes the fold's flag
    panel_finish<T, PR, TB, kTileWaves, 2>(p, acc, rg0, tok0, SK, sk, rt, tt, wave, lane, reinterpret_cast<int *>(win));
}

// Output of an eight-wave panel that is computed whole: every wave turns its 64 rows x 128 tokens around in LDS (the ring
// is free by then; 144 bytes per token, so that the 8-byte pieces of 32 tokens meet each bank at most twice) and stores
// whole 128-byte lines, eight tokens per instruction.  Stored straight from the accumulators, a lane's four rows of one
// token are 8 bytes in a line that fifteen other instructions complete: 67 MB of output took 23 us that way.
constexpr int kP8OutPitch = 144;                               // bytes per token in the turn-around buffer
constexpr size_t kP8OutBytes = (size_t)8 * 128 * kP8OutPitch;
template <class T, int TB>
__device__ __forceinline__ void p8_store_panel(const PanelArgs &p, f32x16 (&acc)[2][TB], int rg0, int tok0, int wave, int lane,
                                               u32x4 *win) {
    uint8_t *buf = reinterpret_cast<uint8_t *>(win) + (size_t)wave * 128 * kP8OutPitch;
    const int half = lane >> 5, c32 = lane & 31;
    const int n0 = rg0 * 16;                                   // first of the wave's 64 rows
#pragma unroll
    for (int pr = 0; pr < 2; ++pr)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int row = pr * 32 + 8 * g + 4 * half;        // of the wave's 64
            float bias[4] = {0.f, 0.f, 0.f, 0.f};
            if (p.bias && n0 + row < p.N) {
#pragma unroll
                for (int i = 0; i < 4; ++i) bias[i] = T::to_f32(p.bias[n0 + row + i]);
            }
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) {
                u32x2 o;
                o[0] = T::from_f32x2(p.alpha * acc[pr][tb][4 * g] + bias[0], p.alpha * acc[pr][tb][4 * g + 1] + bias[1]);
                o[1] = T::from_f32x2(p.alpha * acc[pr][tb][4 * g + 2] + bias[2], p.alpha * acc[pr][tb][4 * g + 3] + bias[3]);
                *reinterpret_cast<u32x2 *>(buf + (tb * 32 + c32) * kP8OutPitch + row * 2) = o;
            }
        }
    // lane 8 t + q: 16 bytes (8 rows) q of token t of each group of eight tokens
    const int t8 = lane >> 3, q = lane & 7;
    const bool rows_ok = n0 + q * 8 < p.N;
#pragma unroll
    for (int it = 0; it < 4 * TB; ++it) {
        const int token = it * 8 + t8;
        const u32x4 v = *reinterpret_cast<const u32x4 *>(buf + token * kP8OutPitch + q * 16);
        if (rows_ok && tok0 + token < p.M) *reinterpret_cast<u32x4 *>(p.C + (size_t)(tok0 + token) * p.N + n0 + q * 8) = v;
    }
}

// ---------------------------------------------------------------------------------------------------------------
// 256 x 256 panels: the eight-wave loop of mlk_panel8.cuh.
//
// Grid: without K slices the workgroup ids of an XCD walk bands of p.band groups of eight row tiles in chunks of
// p.chunk token tiles, so that the 32 workgroups an XCD runs at a time cover 8 x 4 (row tiles x token tiles) and share
// both operands through its L2; with the token tiles of two row tiles side by side (2 x 16) the same product took
// 17 % longer (8192 x 8192, 4096 tokens: 491 against 413 us).  A fifth slab of LDS (160 KiB) changed nothing.
template <class T, bool FP8, int TB>
__device__ __forceinline__ void gemm_panel8(const PanelArgs &p, int rt, int tt, int sk, int SK) {
    extern __shared__ u32x4 win[];
    constexpr int PR = 2;
    constexpr int WBYTES = FP8 ? 1 : 2;
    using Loop = Panel8Loop<T, FP8, TB>;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave & 3, wt = wave >> 2;
    const int groups = p.N >> 4;
    const int rgp = rt * 16;                                   // first row group of the panel
    const int rg0 = rgp + wr * 4;                              // of this wave
    const int tok0 = tt * 256;
    const int nwin_total = p.K / 64;                           // slices are cut in windows of 64 k, as the host counts them
    const int wbeg = (int)((long long)sk * nwin_total / SK);
    const int slab0 = 2 * wbeg;
    const int nslab = 2 * ((int)((long long)(sk + 1) * nwin_total / SK) - wbeg);

    // sources of this wave's loads: weight tiles 2 wave, 2 wave + 1 of the panel (rows past N: a copy of the last row
    // group, never stored), its token chunks (tokens past M: the last token)
    P8Src src;
    src.a = p.A + (size_t)rgp * p.K * 16 * WBYTES;
    src.b = p.B;
    const int rga = min(rgp + 2 * wave, groups - 1), rgb = min(rgp + 2 * wave + 1, groups - 1);
    ScaleRow srow;
    if constexpr (FP8) {
        src.a_off[0] = (uint32_t)((lane >> 5 ? rgb : rga) - rgp) * (uint32_t)p.K * 16u + (lane & 31) * 16;
        const int scale_cols = (p.K + 127) >> 7;
        srow = load_scale_row(p.scale ? p.scale + (size_t)(rga >> 3) * scale_cols : nullptr, scale_cols, lane);
    } else {
        src.a_off[0] = (uint32_t)(rga - rgp) * (uint32_t)p.K * 32u;
        src.a_off[1] = (uint32_t)(rgb - rgp) * (uint32_t)p.K * 32u;
    }
#pragma unroll
    for (int i = 0; i < Loop::NB; ++i) {
        const int tok = min(tok0 + p8_chunk<TB>(wave, i) * 16 + (lane >> 2), p.M - 1);
        src.b_off[i] = (uint32_t)tok * (uint32_t)p.K * 2u + p8_lane_octet(lane);
    }
    f32x16 acc[PR][TB];
    zero_acc(acc);
    Loop::run(acc, src, srow, slab0, nslab, wave, lane);
    __syncthreads();
    if (TB < 4 || SK == 1) p8_store_panel<T, TB>(p, acc, rg0, tok0 + wt * 32 * TB, wave, lane, win);
    else if constexpr (TB == 4)
        panel_finish<T, PR, TB, 8, 2>(p, acc, rg0, tok0 + wt * 128, SK, sk, rt, tt, wave, lane, reinterpret_cast<int *>(win));
}

template <class T, bool FP8>
__global__ void __launch_bounds__(512) gemm_panel8_kernel(PanelArgs p) {
    // workgroup -> (row tile, k slice, token tile), as in gemm_panel_kernel
    const int xcd = blockIdx.x & 7;
    int u = blockIdx.x >> 3;
    int SK, sk, tt, rt;
    if (p.band > 0) {
        const int TT = p.token_tiles, groups8 = (p.row_tiles + 7) >> 3, RB = p.band, TC = p.chunk;
        const int band = u / (RB * TT);
        const int nb = min(RB, groups8 - band * RB);           // groups of row tiles in this band
        const int v = u - band * RB * TT;
        const int c = v / (nb * TC);
        const int tc = min(TC, TT - c * TC);                   // token tiles in this chunk
        const int w = v - c * nb * TC;
        SK = 1, sk = 0;
        tt = c * TC + w % tc;
        rt = (band * RB + w / tc) * 8 + xcd;
    } else {
        const int whole_wgs = p.whole_groups * p.token_tiles;
        const bool sliced = u >= whole_wgs;
        SK = sliced ? p.SK : 1;
        if (sliced) u -= whole_wgs;
        tt = u % p.token_tiles;
        u /= p.token_tiles;
        sk = u % SK;
        rt = ((sliced ? p.whole_groups : 0) + u / SK) * 8 + xcd;
    }
    if (rt >= p.row_tiles) return;
    // The last token tile multiplies the 64, 128 or 192 token columns that cover it (28672 x 4096 bf16 at 700 tokens 196 ->
    // 193 us, 13824 x 5120 at 3000 tokens 372 -> 367 us); the fold of K slices knows whole tiles.
    switch (SK == 1 ? min(4, (p.M - tt * 256 + 63) >> 6) : 4) {
        case 1: gemm_panel8<T, FP8, 1>(p, rt, tt, sk, SK); break;
        case 2: gemm_panel8<T, FP8, 2>(p, rt, tt, sk, SK); break;
        case 3: gemm_panel8<T, FP8, 3>(p, rt, tt, sk, SK); break;
        default: gemm_panel8<T, FP8, 4>(p, rt, tt, sk, SK); break;
    }
}

// Tokens per panel when the caller leaves the choice open.  Workgroups run one per CU in rounds; a 256-token panel
// takes 1.3 to 1.5 times as long as a 128-token one for 16-bit weights (eight-wave kernel) and 1.84 times for soft-FP8
// ones (measured), so the width with the cheaper sum of rounds wins.
int panel_tokens(int m, int n, bool fp8) {
    const int cus = device_cus();
    const long long row_tiles = (n + kPanelRowsPerWg - 1) / kPanelRowsPerWg;
    const long long rounds128 = (row_tiles * ((m + 127) / 128) + cus - 1) / cus;
    const long long rounds256 = (row_tiles * ((m + 255) / 256) + cus - 1) / cus;
    return rounds256 * (fp8 ? 184 : 140) < rounds128 * 100 ? 256 : 128;
}

size_t panel_partial_bytes(int m, int n, int sk) {
    const size_t row_tiles = (n + kPanelRowsPerWg - 1) / kPanelRowsPerWg;
    const size_t tokens = (size_t)((m + 255) / 256) * 256;       // covers both panel widths
    return (size_t)sk * row_tiles * kPanelRowsPerWg * tokens * 4;
}

// a_kind: MLK_F16, MLK_BF16 or MLK_FP8_E4M3 (bf16 activations); width: tokens per panel (128 or 256), anything else =
// panel_tokens(m, n); rows: weight rows per panel (128 or 256; 128 only with 128 tokens), anything else = chosen
// from the number of panels; sk: K slices; last_round_only: slice only the panels that are left over after whole
// rounds of one panel per CU (every panel when there is less than a round, none when nothing is left over or where
// the leftover cannot be told apart and slicing everything costs more)
int launch_panel(const void *a, const void *b, void *c, int m, int n, int k, int a_kind, float alpha, const void *bias,
                 const float *scale, int width, int rows, int sk, bool last_round_only, void *counters,
                 size_t counter_bytes, void *partial, size_t partial_bytes, hipStream_t s) {
    PanelArgs p = {};
    p.A = (const uint8_t *)a;
    p.B = (const uint16_t *)b;
    p.C = (uint16_t *)c;
    p.bias = (const uint16_t *)bias;
    p.scale = scale;
    p.partial = (f32x4 *)partial;
    p.counters = (int *)counters;
    p.M = m;
    p.N = n;
    p.K = k;
    p.alpha = alpha;
    if (width != 128 && width != 256) width = panel_tokens(m, n, a_kind == MLK_FP8_E4M3);
    p.token_tiles = (m + width - 1) / width;
    MLK_REQUIRE(k % 128 == 0, "gemm: the panel kernel needs K % 128 == 0");
    MLK_REQUIRE((long long)m * k < (1ll << 31), "gemm: the panel kernel indexes activations with 32 bits");
    const int windows = k / (panel_kw(width / 32) * 32);
    if (sk > windows) sk = windows;
    if (sk < 1) sk = 1;
    p.SK = sk;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) dev = 0;
    if (width == 256) rows = 256;
    if (rows != 128 && rows != 256) {
        const int cus = device_cus();
        // few panels: 128-row panels put twice as many CUs to work (a 128-row panel takes two thirds of the time of
        // a 256-row one); from three eighths of the CU count on, 256-row panels and K slices fill the chip better
        const long long panels256 = (long long)((n + 255) / 256) * p.token_tiles;
        rows = panels256 * 8 <= (long long)cus * 3 ? 128 : 256;
    }
    p.row_tiles = (n + rows - 1) / rows;
    const int groups = (p.row_tiles + 7) / 8;                 // groups of eight row tiles, one per XCD
    p.whole_groups = 0;
    if (last_round_only && sk > 1) {
        // workgroups start in the order of their ids, eight XCDs taking turns: a round is CUs / 8 workgroups per XCD
        const int per_xcd = device_cus() / 8;
        if (p.token_tiles <= per_xcd && per_xcd % p.token_tiles == 0) {
            const int groups_per_round = per_xcd / p.token_tiles;
            p.whole_groups = groups / groups_per_round * groups_per_round;
        }
        if (p.whole_groups == groups) p.whole_groups = 0, p.SK = sk = 1;    // nothing left over
    }
    if (sk > 1) {
        MLK_REQUIRE(partial != nullptr && counters != nullptr, "gemm: a K split across workgroups needs a workspace");
        MLK_REQUIRE((size_t)p.row_tiles * p.token_tiles * sizeof(int) <= counter_bytes,
                    "gemm: too many panels for the counter region");
        if (partial_bytes < panel_partial_bytes(m, n, sk)) return fail(MLK_ERR_WORKSPACE, "gemm: workspace too small");
    }
    // Token tiles that do not divide an XCD's CUs leave no groups that fill whole rounds, and slicing every panel of a grid of
    // several rounds pays the fold for all of it: then the panels are computed whole, unless the slices save more time in
    // rounds than their partial products cost (written and read once at about 5 TB/s).  Row tiles belong to XCDs, so a round
    // is CUs / 8 workgroups of one XCD, and the fullest XCD counts.
    // 11008 x 4096 fp16 at 2100 tokens (nine tiles): 374 us in two slices, 199 us whole; bf16 at 3300 tokens 495 and 286 us;
    // soft-FP8 28672 x 8192 at 1100 tokens 739 us in three slices, 499 us whole; but soft-FP8 4608 x 7168 at 800 tokens (35
    // panels of 128 x 128 on half of the XCDs) 132 us in four slices, 161 us whole.  Over the 294 grids of this kind that the
    // shipped tables lead to, at their fewest, middle and most tokens, twice, the choice is within 7 % of the better one, and within
    // 3 % on all but 11 of 1764 (rounds counted over the whole chip and a panel's time taken as rows times tokens: up to 53 %).
    // Operands off 16 bytes stay sliced where the whole panels run the loop that loads straight into LDS and the sliced ones do not.
    const bool whole_loads_lds = a_kind == MLK_FP8_E4M3 && width == 128 && rows == 256;
    if (last_round_only && sk > 1 && p.whole_groups == 0 && groups * p.token_tiles > device_cus() / 8 &&
        (!whole_loads_lds || (aligned16(a) && aligned16(b)))) {
        const int per_xcd = groups * p.token_tiles, round = device_cus() / 8;
        // us per k32 slab of a round of panels (whole soft-FP8 panels of 256 x 128 run two per CU: 0.65 us for a full round of
        // those, 0.5 us for half a one), and what a round takes to start and to store: 6 us whole, 2 us sliced and 5 us for the fold
        const double slab_us = width == 256 ? 0.8 : rows == 256 ? 0.57 : a_kind == MLK_FP8_E4M3 ? 0.35 : 0.29;
        const double slabs = k / 32;
        const double whole_rounds = (per_xcd + round - 1) / round, sliced_rounds = (double)(((long long)per_xcd * sk + round - 1) / round);
        double whole_us = whole_rounds * slab_us * slabs;
        if (whole_loads_lds) {
            const int left = per_xcd % (2 * round);
            whole_us = (per_xcd / (2 * round) * 0.65 + (left > round ? 0.65 : left > 0 ? 0.5 : 0.)) * slabs;
        }
        whole_us += whole_rounds * 6;
        const double sliced_us = sliced_rounds * (slab_us * slabs / sk + 2) + (double)sk * m * n * 8 / 5e6 + 5;
        if (whole_us <= sliced_us) p.SK = sk = 1;
    }
    const int grid = (p.whole_groups + (groups - p.whole_groups) * sk) * 8 * p.token_tiles;
    // one workgroup per CU (the register ring and the accumulators take a whole SIMD's file); more than 64 KiB of
    // dynamic LDS has to be requested once per kernel
#define MLK_PANEL(TT, F8, TBB, PRR)                                                                                    \
    do {                                                                                                           \
        const size_t lds = (size_t)3 * panel_win(TBB) * 16;                                                        \
        static bool ready_on[64] = {};                           /* the attribute belongs to a device */          \
        bool &ready = ready_on[dev & 63];                                                                          \
        if (!ready) {                                                                                              \
            hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_panel_kernel<TT, F8, TBB, PRR>),    \
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);             \
            if (e != hipSuccess) return fail(MLK_ERR_LAUNCH, hipGetErrorString(e));                                \
            ready = true;                                                                                          \
        }                                                                                                          \
        gemm_panel_kernel<TT, F8, TBB, PRR><<<grid, 256, lds, s>>>(p);                                                  \
    } while (0)
    if (width == 256) {
        // eight waves, operands through LDS
#define MLK_PANEL8(KERNEL, LDS)                                                                                        \
    do {                                                                                                           \
        static bool ready_on[64] = {};                                                                             \
        bool &ready = ready_on[dev & 63];                                                                          \
        if (!ready) {                                                                                              \
            hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(KERNEL),                            \
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)(LDS));           \
            if (e != hipSuccess) return fail(MLK_ERR_LAUNCH, hipGetErrorString(e));                                \
            ready = true;                                                                                          \
        }                                                                                                          \
        KERNEL<<<grid, 512, LDS, s>>>(p);                                                                          \
    } while (0)
        const bool whole = p.SK == 1 && p.whole_groups == 0;
        p.band = whole ? 8 : 0;
        p.chunk = 4;
        // LDS: the ring, or the turn-around buffer of the output if that is larger
        constexpr size_t lds16 = kP8RingBytes > kP8OutBytes ? kP8RingBytes : kP8OutBytes;
        constexpr size_t lds8 = kP8Fp8LdsBytes > kP8OutBytes ? kP8Fp8LdsBytes : kP8OutBytes;
        if (a_kind == MLK_FP8_E4M3) MLK_PANEL8((gemm_panel8_kernel<BF16, true>), lds8);
        else if (a_kind == MLK_F16) MLK_PANEL8((gemm_panel8_kernel<F16, false>), lds16);
        else MLK_PANEL8((gemm_panel8_kernel<BF16, false>), lds16);
#undef MLK_PANEL8
    } else if (rows == 256 && a_kind == MLK_FP8_E4M3 && (p.SK == 1 || p.whole_groups > 0)) {
        // soft-FP8, panels computed whole (or only the last round's sliced): the loop that prefetches through LDS, two
        // workgroups per CU (28672 x 8192 at 1024 tokens: 616 -> 474 us); fully sliced grids and 16-bit weights stay on
        // the register-ring loop, which was ahead there (compared while the fold of this kernel still spilled)
#define MLK_PANEL_LDS(TT, F8, RING)                                                                                    \
    do {                                                                                                           \
        constexpr size_t lds = PanelLdsShape<F8, 4, RING>::lds_bytes;                                              \
        static bool ready_on[64] = {};                                                                             \
        bool &ready = ready_on[dev & 63];                                                                          \
        if (!ready) {                                                                                              \
            hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_panel_lds_kernel<TT, F8, RING>), \
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);             \
            if (e != hipSuccess) return fail(MLK_ERR_LAUNCH, hipGetErrorString(e));                                \
            ready = true;                                                                                          \
        }                                                                                                          \
        gemm_panel_lds_kernel<TT, F8, RING><<<grid, 256, lds, s>>>(p);                                             \
    } while (0)
        MLK_PANEL_LDS(BF16, true, 4);
#undef MLK_PANEL_LDS
    } else if (rows == 256) {
        if (a_kind == MLK_FP8_E4M3) MLK_PANEL(BF16, true, 4, 2);
        else if (a_kind == MLK_F16) MLK_PANEL(F16, false, 4, 2);
        else MLK_PANEL(BF16, false, 4, 2);
    } else {
        if (a_kind == MLK_FP8_E4M3) MLK_PANEL(BF16, true, 4, 1);
        else if (a_kind == MLK_F16) MLK_PANEL(F16, false, 4, 1);
        else MLK_PANEL(BF16, false, 4, 1);
    }
#undef MLK_PANEL
    MLK_LAUNCH_CHECK();
    return MLK_OK;
}

}  // namespace mlk
