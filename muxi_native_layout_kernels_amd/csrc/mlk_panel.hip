// Kernel ids 3 and 5: panel GeMM for more than 64 tokens over layout-A weights (row-major activations and
// output), where the product is bound by the matrix cores and no longer by the weight stream; and the launch plan and entry of kernel
// id 8 (mlk_panel8_gemm.cuh), which serves calls that name no launch parameters.  Calls and table rows that ask for ids 3 and 5 run
// here, and operands off 16 bytes above 64 tokens (gemm_plan_off16).
//
// A workgroup of four waves computes a panel of 256 weight rows x 128 tokens over one of SK slices
// of K with v_mfma_f32_32x32x16 (one wave per SIMD issues the 16x16x32 form at little more than half
// rate; the 32x32 form runs at nine tenths of peak from a single wave).  Every wave owns four row
// groups (two pairs of 32 rows) and all four blocks of 32 tokens: eight 32x32 accumulators.  Two other
// shapes exist: 256 rows x 256 tokens (the eight-wave panels of mlk_panel8_gemm.cuh) when that
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
#include <math.h>

#include "mlk_panel_loop.cuh"
#include "mlk_panel8_gemm.cuh"

namespace mlk {

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

    panel_finish<T, PR, TB, TB>(p, acc, rg0, tok0, SK, sk, rt, tt, wave, lane, &s_last);
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
    panel_finish<T, PR, TB, 2>(p, acc, rg0, tok0, SK, sk, rt, tt, wave, lane, reinterpret_cast<int *>(win));
}

extern template int launch_panel8<BF16, false>(const Panel8Args &, int, int, hipStream_t);
extern template int launch_panel8<F16, false>(const Panel8Args &, int, int, hipStream_t);
extern template int launch_panel8<BF16, true>(const Panel8Args &, int, int, hipStream_t);

// Lines, whole and dealt panels of m x n x k in panels of 128 pr rows x 64 tb tokens.  sk = 1: every panel whole; from 2 on: in that
// many slices of K; kP8Deal: dealt evenly to one workgroup per CU.  With more panels than CUs only those that are left over after
// whole rounds of one panel per CU are sliced or dealt, unless the caller says how many groups of eight row tiles are not (kernel ids
// 3 and 5 on panels of 256 x 256).
// kP8Deal is no count that a caller can ask for: kernel id 8 says it as p3 = 64, but ids 3 and 5 take p3 = 64 for as many slices, and
// their workspace holds those.
constexpr int kP8Deal = 1 << 20, kP8DealP3 = 64;
static void panel8_shape(Panel8Args &p, int m, int n, int k, int pr, int tb, int sk, int whole_groups = -1) {
    const int cus = device_cus(), windows = k / 64;
    p.M = m;
    p.N = n;
    p.K = k;
    p.row_tiles = (n + 128 * pr - 1) / (128 * pr);
    p.token_tiles = (m + 64 * tb - 1) / (64 * tb);
    p.cols = p.token_tiles == 1 ? (m + 15) / 16 * 16 : 64 * tb;
    const int panels = p.row_tiles * p.token_tiles;
    const bool bands = whole_groups > 0 || (whole_groups < 0 || sk <= 1 ? panels > cus : false);
    p.band = bands ? 8 : 0;
    p.chunk = 4;
    p.panels = bands ? (p.row_tiles + 7) / 8 * p.token_tiles : panels;
    p.whole = p.panels;
    p.deal = 0;
    p.slots = 1;
    if (sk <= 1) return;
    const int round = bands ? cus / 8 : cus;                 // workgroups of a line that run at a time
    const int whole = whole_groups >= 0 ? whole_groups * p.token_tiles : (bands ? p.panels / round * round : 0), rest = p.panels - whole;
    if (rest == 0) return;
    p.whole = whole;
    if (sk != kP8Deal) {
        p.deal = rest * (sk < windows ? sk : windows);
    } else {
        p.deal = round < rest * windows ? round : rest * windows;
        p.slots = 2;
    }
}
static size_t panel8_partial_bytes(const Panel8Args &p, int pr) {
    return (size_t)(p.band > 0 ? 8 : 1) * p.deal * p.slots * pr * p.cols * 512;
}
// p3: as kernel id 8 takes it
static int panel8_slices(int p3) { return p3 == kP8DealP3 ? kP8Deal : p3; }
size_t panel8_partial_bytes(int m, int n, int k, int pr, int tb, int p3) {
    Panel8Args p = {};
    panel8_shape(p, m, n, k, pr, tb, panel8_slices(p3));
    return panel8_partial_bytes(p, pr);
}

size_t panel_partial_bytes(int m, int n, int sk) {
    const size_t row_tiles = (n + kPanelRowsPerWg - 1) / kPanelRowsPerWg;
    const size_t tokens = (size_t)((m + 255) / 256) * 256;       // covers both panel widths
    return (size_t)sk * row_tiles * kPanelRowsPerWg * tokens * 4;
}

// Time in us that m x n x k takes in panels of 128 pr rows x 64 tb tokens with K in sk slices (kP8Deal: only for grids of several
// rounds).  Fitted to the times of 1449 products (512 to 37888 rows, K 512 to 18432, 65 to 4096 tokens; bf16 and soft-FP8, the 9 to 14 likeliest
// launches of each), to the times and to how much slower than the best the launch is that it picks.  Each launch was timed twice, on weights that come from
// memory and on two copies in turn, which the Infinity Cache holds up to 128 MB: they rank launches differently (11008 x 4096 bf16 at 128 tokens, panels of
// 128 x 64 whole and 128 x 128 in two slices: 35.6 and 33.4 us from memory, 24.8 and 27.1 from the cache), and what is fitted is the geometric mean
// of both.  On as many other products the launch it picks is 0.8 % (soft-FP8 0.5 %) slower than the best one in the geometric mean, 4.1 % (2.8 %) at
// the 95th percentile (1.1 % and 6 % from memory or from the cache alone); a margin of 2 to 5 % in favour of launches in one slice picks no better.
// What it does not know: panels of one row tile are faster where one token tile is shorter than the others, which runs ahead and fetches
// their weights (11008 x 4096 at 300 tokens in panels of 128 x 192: 192 and 108 tokens 44.0 us, 160 and 140 45.6); and that a count of
// slices can be a fifth slower than the next one (512 x 2176 at 446 tokens in four and five: 11.9 and 14.4).
struct P8Cost {
    // up to one panel per CU: start, store (256 x 256), fold = fold + fold_slice per slice + fold_mb per MB of slots; a k32 slab of a panel
    // on an idle chip, what a workgroup on every CU adds to it, and the power of the token tiles that share weights by which that falls
    float start, store, fold, fold_slice, fold_mb, shared, slab[2][4], busy[2][4];
    // several rounds: start, end of a round (256 x 256), what a last round that is not full saves of its empty part, fold, per MB; a slab
    float r_start, r_end, r_empty, r_fold, r_fold_mb, r_slab[2][4];
};
static const P8Cost kP8Cost16 = {3.343f, 4.509f, 3.000f, 0.143f, 0.292f, 0.501f,
                                 {{0.140f, 0.199f, 0.258f, 0.355f}, {0.224f, 0.297f, 0.395f, 0.515f}},
                                 {{0.102f, 0.110f, 0.107f, 0.083f}, {0.269f, 0.287f, 0.204f, 0.228f}},
                                 2.969f, 5.880f, 0.250f, 3.548f, 0.574f,
                                 {{0.205f, 0.287f, 0.339f, 0.426f}, {0.354f, 0.427f, 0.554f, 0.666f}}};
static const P8Cost kP8Cost8 = {5.004f, 4.579f, 3.301f, 0.115f, 0.254f, 0.021f,
                                {{0.132f, 0.179f, 0.265f, 0.317f}, {0.219f, 0.279f, 0.436f, 0.515f}},
                                {{0.050f, 0.080f, 0.076f, 0.096f}, {0.103f, 0.187f, 0.198f, 0.166f}},
                                3.996f, 9.576f, 0.208f, 3.131f, 0.384f,
                                {{0.181f, 0.275f, 0.362f, 0.429f}, {0.351f, 0.451f, 0.613f, 0.649f}}};
// Up to 64 tokens, where panels of 64 compete with the narrow kernels: fitted to 430 products of 16 to 64 tokens, timed in the same way, with the
// times that narrow_us() expects beside them.  On as many others the choice between all is 5.0 % (soft-FP8 3.7 %) slower than the best, with the constants of the
// loops before the 16 x 16 products 5.3 % (4.2 %): what is left is in the narrow kernels.
static const P8Cost kP8Few16 = {3.446f, 2.918f, 3.334f, 0.101f, 0.269f, 0.f, {{0.121f}, {0.165f}}, {{0.157f}, {0.405f}},
                                4.762f, 7.372f, 0.463f, 3.750f, 0.248f, {{0.286f}, {0.315f}}};
static const P8Cost kP8Few8 = {4.351f, 2.866f, 3.136f, 0.094f, 0.259f, 0.f, {{0.137f}, {0.224f}}, {{0.056f}, {0.163f}},
                               5.817f, 8.709f, 0.468f, 4.593f, 0.197f, {{0.207f}, {0.322f}}};
static double panel8_us(const P8Cost &f, int m, int n, int k, int pr, int tb, int sk) {
    const int cus = device_cus(), rows = (n + 128 * pr - 1) / (128 * pr), tokens = (m + 64 * tb - 1) / (64 * tb), windows = k / 64;
    const int narrow = (m - (tokens - 1) * 64 * tb + 63) / 64;                   // columns / 64 of the last token tile
    const long long panels = (long long)rows * tokens;
    if (panels <= cus) {
        const int t = tokens == 1 ? narrow : tb;
        const double wgs = (double)panels * sk, busy = wgs < cus ? wgs / cus : 1;
        const double slab = f.slab[pr - 1][t - 1] + f.busy[pr - 1][t - 1] * busy * pow(tokens, -f.shared);
        double us = f.start + f.store * pr * t / 8 + 2 * ((windows + sk - 1) / sk) * slab;
        if (sk > 1) us += f.fold + f.fold_slice * sk + f.fold_mb * wgs * pr * t * 0.032768;
        return us;
    }
    // row tiles belong to XCDs, and the fullest one counts
    const int groups = (rows + 7) / 8, round = cus / 8;
    const long long per_xcd = (long long)groups * tokens, rounds = (per_xcd + round - 1) / round;
    const long long full = (long long)groups * (narrow < tb ? tokens - 1 : tokens);              // panels of all 64 tb columns
    const double slabs = 2. * windows, end = f.r_end * pr * tb / 8;
    const double t_full = f.r_slab[pr - 1][tb - 1] * slabs, t_narrow = f.r_slab[pr - 1][narrow - 1] * slabs;
    const double even = (full * t_full + (per_xcd - full) * t_narrow) / round;                   // dealt out evenly
    if (sk == 1) {
        // The last round is as long as a full panel unless the narrow ones are all that it holds: they stand alone at the end where the last chunk
        // of token tiles is theirs (11008 x 4096 at 1302 tokens in panels of 256 x 256, 36 on the fullest XCD: 159 us, priced as narrow 125, dealt 116).
        const long long last = per_xcd - round * (rounds - 1);
        const bool narrow_last = narrow < tb && last <= ((tokens - 1) % 4 ? 1 : (groups - 1) % 8 + 1);
        const double dealt = even + (double)per_xcd / round * end;
        const double whole = (rounds - 1) * t_full + (narrow_last ? t_narrow : t_full) + rounds * end;
        return f.r_start + dealt + (whole - dealt) * (1 - f.r_empty);
    }
    const long long rest = per_xcd % round;
    if (rest == 0) return 1e30;                                                                  // nothing is left over
    // XCDs that have one group of row tiles less deal less, or nothing
    const int most = rows - 8 * (groups - 1);
    const double lines = most + (8 - most) * (rest > tokens ? (double)(rest - tokens) / rest : 0);
    // 3 % in favour of whole panels, which are as good where the two come out alike
    return 1.03 * (f.r_start + even + (per_xcd / round + 1.2) * end + f.r_fold + f.r_fold_mb * round * lines * pr * tb * 0.032768);
}

// Time in us of the narrow kernels (ids 1 and 4) on up to 64 tokens: what a CU pulls through its memory path (weights, and the
// activations of every workgroup on it), the weight stream of the whole chip, and the chain of one wave's k tiles, whichever is longest,
// then the fold of K slices; a little more for more waves and, with several workgroups on a CU, for large ones.  Fitted per count of token
// blocks (one, two, three and four) to 31 weight shapes outside the tables (640 to 38400 rows, K 512 to 14336) at up to eight token
// counts, 8000 launches: the choice is 4 % above the best of some thirty launches per shape, panels included (geometric mean), and 1.34 times
// as fast as the fixed launch parameters it replaces.
struct NarrowCost {
    float weight_line, token_line, tile, start, fold, fold_mb, product, crowd, stream, even, staged, waves, crowd_rows;
};
static const NarrowCost kNarrow16[3] = {
    {2.674f, 3.245f, 0.103f, 3.192f, 1.750f, 0.690f, 0.f, 0.032f, 6.798f, 1.042f, 1.f, 0.011f, 0.037f},
    {2.823f, 3.157f, 0.001f, 3.559f, 1.402f, 0.884f, 0.037f, 0.008f, 6.104f, 1.026f, 1.067f, 0.f, 0.026f},
    {3.249f, 1.903f, 0.222f, 4.343f, 1.447f, 1.188f, 0.017f, 0.002f, 6.232f, 1.018f, 0.949f, 0.025f, 0.f}};
static const NarrowCost kNarrow8[3] = {
    {3.428f, 2.427f, 0.107f, 3.792f, 1.888f, 0.447f, 0.016f, 0.062f, 5.710f, 1.f, 1.f, 0.016f, 0.011f},
    {3.388f, 3.051f, 0.001f, 3.867f, 1.530f, 0.798f, 0.042f, 0.f, 6.150f, 1.296f, 0.802f, 0.011f, 0.037f},
    {5.594f, 1.576f, 0.257f, 4.918f, 1.034f, 1.046f, 0.019f, 0.f, 5.555f, 1.063f, 0.734f, 0.036f, 0.f}};
static double narrow_us(bool fp8, int m, int n, int k, int id, int p1, int p2, int p3) {
    const int blocks = (m + 15) / 16, groups = n / 16, cus = device_cus(), size = fp8 ? 1 : 2;
    const NarrowCost &f = (fp8 ? kNarrow8 : kNarrow16)[blocks > 2 ? 2 : blocks - 1];
    const int rows = id == 4 ? (groups + cus - 1) / cus : p1;                            // row groups of a workgroup
    const int wgs = id == 4 ? cus : (groups + p1 - 1) / p1 * p3;
    const double per = id == 4 ? 1 : wgs <= 2 * cus ? (wgs + cus - 1) / cus : (double)wgs / cus + 0.35;
    const double depth = (double)k / p3, staged = id == 4 && blocks > 1 ? f.staged : 1;
    const double pull = per * (f.weight_line * rows * 16 * depth * size / 128 + f.token_line * staged * m * depth * 2 / 128) / 1000;
    const double stream = (double)n * k * size / (f.stream * 1e6), load = pull > stream ? pull : stream;
    const double waves = per * p2 / 16, chain = depth / 32 / p2 * (f.tile + f.product * rows * blocks) * (waves > 1 ? waves : 1);
    double us = f.start + sqrt(sqrt(load * load * load * load + chain * chain * chain * chain));
    if (p3 > 1) us += f.fold + f.fold_mb * p3 * n * m * 4e-6;
    const double octaves = log2((double)p2) - 2;
    us *= 1 + f.waves * octaves + (id != 4 && per > 1 ? f.crowd * octaves : 0) + (id != 4 && per > 1.5 ? f.crowd_rows * log2((double)rows) : 0);
    return id == 4 ? us * f.even : us;
}

// Launches of the narrow kernels (ids 1 and 4) for up to 64 tokens, whose partial sums of K slices take at most `row_blocks` KiB per
// token block.
template <class Offer>
static void narrow_offers(int m, int n, int k, bool fp8, bool b_native, size_t row_blocks, Offer offer) {
    const int groups = n / 16, cus = device_cus();
    // the plain launch: two row groups up to 32 tokens, waves until the chip has eight per CU; 4 % in its favour
    int r = m > 32 || groups % 2 ? 1 : 2, waves = 1;
    while (waves < 16 && (long long)groups / r * waves < 8 * cus) waves *= 2;
    offer(0.96 * narrow_us(fp8, m, n, k, 1, r, waves, 1), 1, r, waves, 1);
    // kernel 4 exists from two token blocks on with soft-FP8 weights and with layout-B activations
    if (groups > cus && groups <= cus * (fp8 ? 8 : 4) && ((!fp8 && !b_native) || m > 16))
        for (int p2 = 4; p2 <= 8; p2 *= 2) offer(narrow_us(fp8, m, n, k, 4, 1, p2, 1), 4, 1, p2, 1);
    for (int p1 = 1; p1 <= 4; p1 *= 2)
        for (int p2 = 4; groups % p1 == 0 && p2 <= 16; p2 *= 2)
            for (int p3 = 1; p3 <= 8; p3 *= 2)
                if (groups / p1 * (long long)p3 <= 4 * cus && (p3 == 1 || (groups / p1 <= 300 && (size_t)p3 * groups <= row_blocks)) && k / 32 / p3 / p2 >= 1)
                    offer(narrow_us(fp8, m, n, k, 1, p1, p2, p3), 1, p1, p2, p3);
}

// A grid of one line is cut into eight runs, one per XCD, and every XCD fetches what its run reads.  With the token tiles of a row tile
// side by side (the weights then come once) up to eight of them fetch all activations, with the row tiles of a token tile side by
// side all weights.  The order that fetches less, where the activations are the larger operand: 640 x 14464 at 3065 tokens, panels
// of 128 x 256 in four slices, 92 -> 68 us (462 -> 237 MB), 1024 x 5504 at 1623, 128 x 192 in three, 41 -> 34 (154 -> 108); against the
// rule 512 x 7168 at 600, 128 x 64 in six, 15.6 -> 18.9 (42 -> 67).
static bool p8_rows_first(const Panel8Args &p, int m, int n, int k, bool fp8) {
    if (p.band > 0) return false;
    const double weights = (double)n * k * (fp8 ? 1 : 2), tokens = (double)m * k * 2;
    const int rows8 = p.row_tiles < 8 ? p.row_tiles : 8, tokens8 = p.token_tiles < 8 ? p.token_tiles : 8;
    return tokens > weights && tokens + weights * tokens8 < weights + tokens * rows8;
}

// Launch parameters (kernel id, p1, p2, p3) that are expected to be fastest for m tokens x n rows x k.
void gemm_plan(int m, int n, int k, bool fp8, bool b_native, int32_t *out) {
    const P8Cost &f = m <= 64 ? (fp8 ? kP8Few8 : kP8Few16) : fp8 ? kP8Cost8 : kP8Cost16;
    double best = 1e30;
    auto offer = [&](double us, int id, int p1, int p2, int p3) {
        if (us < best) best = us, out[0] = id, out[1] = p1, out[2] = p2, out[3] = p3;
    };
    for (int pr = 1; pr <= 2; ++pr)
        for (int tb = 1; tb <= 4; ++tb) {
            if (tb > 1 && m <= 64 * (tb - 1)) break;
            const long long panels = (long long)((n + 128 * pr - 1) / (128 * pr)) * ((m + 64 * tb - 1) / (64 * tb));
            offer(panel8_us(f, m, n, k, pr, tb, 1), 8, 2 * pr, tb, 1);
            if (panels > device_cus()) offer(panel8_us(f, m, n, k, pr, tb, kP8Deal), 8, 2 * pr, tb, kP8DealP3);
            else
                // slices of at least four slabs that one workgroup per CU takes
                for (int sk = 2; sk <= 32 && panels * sk <= device_cus() && k / 64 / sk >= 2; ++sk)
                    offer(panel8_us(f, m, n, k, pr, tb, sk), 8, 2 * pr, tb, sk);
        }
    if (m <= 64) narrow_offers(m, n, k, fp8, b_native, (size_t)-1, offer);
}

// The same for operands that the panels cannot take (off 16 bytes), with up to `partial_bytes` of partial sums: kernel id 3 on
// row-major operands above 64 tokens, else ids 1 and 4, in passes of up to 64 tokens.
void gemm_plan_off16(int m, int n, int k, bool fp8, bool b_native, bool c_native, size_t partial_bytes, int32_t *out) {
    double best = 1e30;
    out[0] = 1, out[1] = 1, out[2] = 4, out[3] = 1;
    auto offer = [&](double us, int id, int p1, int p2, int p3) {
        if (us < best) best = us, out[0] = id, out[1] = p1, out[2] = p2, out[3] = p3;
    };
    if (m <= 64 || b_native || c_native) {
        const int blocks = (m + 15) / 16;                      // the kernels ask for sums of up to eight token blocks
        narrow_offers(m < 64 ? m : 64, n, k, fp8, b_native, partial_bytes / 1024 / (blocks < 8 ? blocks : 8), offer);
        return;
    }
    // 128-row panels put twice as many CUs to work while there are few; K slices of four windows at least that one workgroup per CU
    // takes
    const int cus = device_cus();
    const long long tokens = (m + 127) / 128;
    const bool small = (n + 255) / 256 * tokens * 8 <= (long long)cus * 3;
    const long long panels = (small ? (n + 127) / 128 : (n + 255) / 256) * tokens;
    int sk = 4;
    while (sk > 1 && (panels * sk > cus || k / 128 / sk < 4 || panel_partial_bytes(m, n, sk) > partial_bytes)) sk >>= 1;
    out[0] = 3, out[1] = small ? 2 : 4, out[2] = 1, out[3] = sk;
}

// whole_groups < 0: kernel id 8, p3 as it takes it; else kernel ids 3 and 5, p3 = K slices of the row tiles behind those groups
int launch_panel8_gemm(const void *a, const void *b, void *c, int m, int n, int k, int a_kind, bool b_native, bool c_native,
                       float alpha, const void *bias, const float *scale, int pr, int tb, int p3, int whole_groups, void *partial,
                       size_t partial_bytes, hipStream_t s) {
    MLK_REQUIRE(k % 128 == 0, "gemm: the panel kernel needs K % 128 == 0");
    MLK_REQUIRE((long long)m * k < (1ll << 31), "gemm: the panel kernel indexes activations with 32 bits");
    Panel8Args p = {};
    p.A = (const uint8_t *)a;
    p.B = (const uint16_t *)b;
    p.C = (uint16_t *)c;
    p.bias = (const uint16_t *)bias;
    p.scale = scale;
    p.partial = (f32x4 *)partial;
    p.alpha = alpha;
    p.b_native = b_native;
    p.c_native = c_native;
    panel8_shape(p, m, n, k, pr, tb, whole_groups < 0 ? panel8_slices(p3) : p3, whole_groups);
    p.rows_first = p8_rows_first(p, m, n, k, a_kind == MLK_FP8_E4M3);
    if (p.deal > 0) {
        MLK_REQUIRE(partial != nullptr, "gemm: a K split across workgroups needs a workspace");
        if (partial_bytes < panel8_partial_bytes(p, pr)) return fail(MLK_ERR_WORKSPACE, "gemm: workspace too small");
    }
    if (a_kind == MLK_FP8_E4M3) return launch_panel8<BF16, true>(p, pr, tb, s);
    if (a_kind == MLK_F16) return launch_panel8<F16, false>(p, pr, tb, s);
    return launch_panel8<BF16, false>(p, pr, tb, s);
}

// Tokens per panel when the caller leaves the choice open.  Workgroups run one per CU in rounds; a round of 256-token panels (eight-wave
// kernel) takes 1.35 to 1.6 times as long as one of 128-token panels, and the width with the cheaper sum of rounds wins.  On 500 products of
// 129 to 4096 tokens, both widths timed, the choice is 1.9 % (soft-FP8 1.2 %) slower than the better one in the geometric mean, the same
// with any ratio from 1 to 1.4; soft-FP8 weights with the 1.84 of an earlier loop: 2.3 %.
int panel_tokens(int m, int n) {
    const int cus = device_cus();
    const long long row_tiles = (n + kPanelRowsPerWg - 1) / kPanelRowsPerWg;
    const long long rounds128 = (row_tiles * ((m + 127) / 128) + cus - 1) / cus;
    const long long rounds256 = (row_tiles * ((m + 255) / 256) + cus - 1) / cus;
    return rounds256 * 140 < rounds128 * 100 ? 256 : 128;
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
    if (width != 128 && width != 256) width = panel_tokens(m, n);
    if (width == 256) rows = 256;
    // the loops that fetch straight into LDS take operands on 16 bytes, and panels of 256 tokens store 16 bytes at a time; others
    // run panels of 128 tokens that fetch through registers
    const bool loads_on16 = aligned16(a) && aligned16(b);
    const bool narrowed = width == 256 && !(loads_on16 && aligned16(c) && aligned16(partial));
    if (narrowed) width = 128;
    p.token_tiles = (m + width - 1) / width;
    MLK_REQUIRE(k % 128 == 0, "gemm: the panel kernel needs K % 128 == 0");
    MLK_REQUIRE((long long)m * k < (1ll << 31), "gemm: the panel kernel indexes activations with 32 bits");
    const int windows = k / (panel_kw(width / 32) * 32);
    if (sk > windows) sk = windows;
    if (sk < 1) sk = 1;
    p.SK = sk;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) dev = 0;
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
    // twice as many panels as the call asked for may be more than have a counter
    if (narrowed && (size_t)p.row_tiles * p.token_tiles * sizeof(int) > counter_bytes) p.whole_groups = 0, p.SK = sk = 1;
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
    // panels of 128 x 128 on half of the XCDs) 132 us in four slices, 161 us whole.  Over 294 grids of this kind (weight
    // shapes of the tables, 65 to 4096 tokens), each at three token counts, twice, the choice is within 7 % of the better one, and within
    // 3 % on all but 11 of 1764 (rounds counted over the whole chip and a panel's time taken as rows times tokens: up to 53 %).
    // Operands off 16 bytes stay sliced where the whole panels run the loop that loads straight into LDS and the sliced ones do not.
    const bool whole_loads_lds = a_kind == MLK_FP8_E4M3 && width == 128 && rows == 256;
    if (last_round_only && sk > 1 && p.whole_groups == 0 && groups * p.token_tiles > device_cus() / 8 && (!whole_loads_lds || loads_on16)) {
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
    if (width == 256)
        return launch_panel8_gemm(a, b, c, m, n, k, a_kind, false, false, alpha, bias, scale, 2, 4, p.SK, p.whole_groups, partial,
                                  partial_bytes, s);
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
    if (rows == 256 && a_kind == MLK_FP8_E4M3 && (p.SK == 1 || p.whole_groups > 0) && loads_on16) {
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
