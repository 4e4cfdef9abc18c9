// Main loops of the eight-wave panels: 128 PR weight rows x 64 TB tokens (PR = 1, 2; TB = 1..4), both operands through LDS,
// fetched with loads that write LDS directly.  Panel8Loop16 is for 16-bit weights (v_mfma_f32_16x16x32), Panel8LoopFp8 for the large
// soft-FP8 panels (16x16x32 with 128 rows, 32x32x16 with 256), Panel8SmallFp8 (mlk_panel8_small.cuh, 32x32x16) for the others;
// Panel8<..>::Loop picks.
//
// What sets the pace of a large panel, measured on 8192 x 8192 bf16 at 4096 tokens (256 x 256 panels, one workgroup per CU; a k32 slab
// takes 0.43 us of products):
//   power    with random operands the clock falls until the card is inside its limit.  A loop of products alone sustains 2.06 PFLOP/s
//            of v_mfma_f32_16x16x32 and 1.80 of 32x32x16 (with zeros 2.47 of both): per operation the 32 x 32 form moves twice as
//            many accumulators through the register file.
//   loads    tokens fetched 32 k at a time are pieces of 64 bytes, and a CU pulls those at half the rate of whole lines: with them
//            the product took 416 us even on zeros.  Fetched 64 k at a time, 342 us; with the weights five slabs deep instead of four and
//            the compiler free to order a slab's instructions, 287 us (products alone: 250 us).
// Together: 430 -> 377 us on random operands; 128 panels of K 14336 (half of the CUs, nothing held back by power) 312 -> 248 us.
// Tried in a copy: weights straight into registers in place of LDS (every weight is then fetched by two waves: 428 us); four waves of
// 128 x 128 (376 us; a third less LDS traffic, but every load stalls the only wave of its SIMD); weights touched ahead into L2,
// token tiles out of step in k, rings deeper than five slabs: within 2 %.
//
// Both waves of a SIMD have to stay inside 256 registers, so nothing is staged through registers: weight tiles (16 rows x 32 k as they
// lie in layout A) are addressed by the thread id alone (the descriptor adds 16 bytes per lane, no address register), tokens come in
// chunks of 8 tokens x 64 k with a per-lane offset (P8TokenPairs).  Wave w = (token half w / 4, row quarter w % 4) multiplies 32 PR
// rows x 32 TB tokens: 2 PR row tiles x 2 TB blocks of 16 tokens.  The barrier is the bare instruction: the fence that comes with
// __syncthreads() would wait for every load in flight.
#pragma once

#include <type_traits>

#include "mlk_panel_lds.cuh"

namespace mlk {

constexpr size_t kP8MostLds = 152 * 1024;                      // of a ring

// Where a wave's loads come from.  A loop says which weight tiles and which tokens a wave fetches: tile(wave, i) for i < PR (16-bit),
// pair(wave): the two tiles 2 pair, 2 pair + 1 (soft-FP8); token(wave, i, lane) and octet(wave, i, lane), the 8 k of a pair of
// slabs, for i < NB; and scale_tile(wave): the first tile of the rows that its (first) row of block scales belongs to.
struct P8Src {
    const uint8_t *a;      // workgroup-uniform base of the weight tiles
    uint32_t a_off[2];     // 16-bit: wave-uniform byte offsets of the wave's PR tiles at k = 0; fp8: [0] = per-lane byte
                           // offset (lanes 0..31 the first tile, 32..63 the second, 16 bytes each)
    const uint16_t *b;     // base of the token rows
    uint32_t b_off[4];     // per-lane byte offsets of this lane's 16 bytes of the wave's chunks at k = 0
    uint32_t b_step;       // bytes from one pair of slabs to the next: of a token row, or of all tokens in layout B
    bool b_runs;           // layout B
};

// The sums of a wave, its 32 PR rows x 32 TB tokens, as its loop leaves them.  each(lane, rows, f): f(row, token, the sums of rows row ..
// row + 3), and rows(row) once ahead of the tokens of four rows; each_half(lane, f), PR = 2: f(row, token, sums of rows row .. + 3,
// sums of rows 32 + row .. + 3).
template <int PR, int TB>
struct P8Acc16 {
    f32x4 acc[2 * PR][2 * TB];                                 // v_mfma_f32_16x16x32: row tiles, blocks of 16 tokens
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int i = 0; i < 2 * PR; ++i)
#pragma unroll
            for (int j = 0; j < 2 * TB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    template <class R, class F>
    __device__ __forceinline__ void each(int lane, R rows, F f) const {
#pragma unroll
        for (int i = 0; i < 2 * PR; ++i) {
            rows(16 * i + 4 * (lane >> 4));
#pragma unroll
            for (int j = 0; j < 2 * TB; ++j) f(16 * i + 4 * (lane >> 4), 16 * j + (lane & 15), acc[i][j]);
        }
    }
    template <class F>
    __device__ __forceinline__ void each_half(int lane, F f) const {
#pragma unroll
        for (int j = 0; j < 2 * TB; ++j)
#pragma unroll
            for (int i = 0; i < 2; ++i) f(16 * i + 4 * (lane >> 4), 16 * j + (lane & 15), acc[i][j], acc[2 + i][j]);
    }
};
template <int PR, int TB>
struct P8Acc32 {
    f32x16 acc[PR][TB];                                        // v_mfma_f32_32x32x16: row pairs, blocks of 32 tokens
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int pr = 0; pr < PR; ++pr)
#pragma unroll
            for (int tb = 0; tb < TB; ++tb)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[pr][tb][e] = 0.f;
    }
    __device__ static __forceinline__ f32x4 quad(const f32x16 &v, int g) { return f32x4{v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]}; }
    template <class R, class F>
    __device__ __forceinline__ void each(int lane, R rows, F f) const {
#pragma unroll
        for (int pr = 0; pr < PR; ++pr)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                rows(32 * pr + 8 * g + 4 * (lane >> 5));
#pragma unroll
                for (int tb = 0; tb < TB; ++tb) f(32 * pr + 8 * g + 4 * (lane >> 5), 32 * tb + (lane & 31), quad(acc[pr][tb], g));
            }
    }
    template <class F>
    __device__ __forceinline__ void each_half(int lane, F f) const {
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
            for (int g = 0; g < 4; ++g) f(8 * g + 4 * (lane >> 5), 32 * tb + (lane & 31), quad(acc[0][tb], g), quad(acc[1][tb], g));
    }
};

// Tokens of two slabs: chunks of 8 tokens x 64 k (128 bytes of a token row, a whole line), TB per wave.  Lane 8 r + j of a chunk's load
// fetches octet j ^ x of token t = r ^ (chunk & 1).  A read of 16 bytes per lane is served for lanes 0..3, 12..15 and 20..27 together, then
// for 4..11, 16..19 and 28..31, and the upper half alike; x is chosen so that those sixteen meet sixteen different bank groups: t for operands of
// 32 tokens; for operands of 16 (F16), where lanes 16..31 hold the next octet, t ^ 1 for the tokens 4..11 of a block (with t, every read took
// twice its time: SQ_LDS_BANK_CONFLICT 2.7e7 in 13824 x 5120 at 3000 tokens).  Activations in
// layout B lie as operands already: a chunk is one run of 1 KiB, 16 tokens of one slab, block j of slab e chunk 2 j + e.  (What a CU
// pulls out of L2: 125 GB/s in runs of 1 KiB, 78 GB/s of loads that gather two pieces or more.)
template <int TB, bool F16>
struct P8TokenPairs {
    static constexpr int NB = TB, B_PAIR = 512 * TB;                    // granules of a pair of slabs
    // x of token t of a chunk c (its parity)
    __device__ static __forceinline__ int swizzle(int t, int c) { return F16 ? t ^ (((t >> 2) ^ c) & 1) : t; }
    __device__ static __forceinline__ int chunk(int wave, int i) { return wave * TB + i; }
    __device__ static __forceinline__ int token_in_chunk(int wave, int i, int lane) { return (lane >> 3) ^ (chunk(wave, i) & 1); }
    __device__ static __forceinline__ int token(int wave, int i, int lane) { return chunk(wave, i) * 8 + token_in_chunk(wave, i, lane); }
    __device__ static __forceinline__ int octet(int wave, int i, int lane) { return (lane & 7) ^ swizzle(token_in_chunk(wave, i, lane), chunk(wave, i) & 1); }
    // Granules of a wave's operands; block j of 16 tokens is at + 128 j.
    // 16x16x32: token lane % 16, octet lane / 16 of slab e.
    __device__ static __forceinline__ int operand16(const P8Src &src, int e, int lane) {
        if (src.b_runs) return 64 * e + lane;
        const int t = lane & 7, c = (lane >> 3) & 1;
        return c * 64 + (t ^ c) * 8 + (((lane >> 4) + 4 * e) ^ swizzle(t, c));
    }
    // 32x32x16: token lane % 32 of a block of 32, octet 2 h + lane / 32 of the pair
    __device__ static __forceinline__ int operand32(const P8Src &src, int h, int lane) {
        const int i = lane & 31, t = i & 7, c = i >> 3;
        if (src.b_runs) return (c >> 1) * 128 + 32 * h + (lane >> 5) * 16 + (i & 15);
        return c * 64 + (t ^ (c & 1)) * 8 + ((2 * h + (lane >> 5)) ^ swizzle(t, c & 1));
    }
    __device__ static __forceinline__ void issue1(const P8Src &src, int wave, u32x4 *dst, int pair, int i) {
        __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)src.b, 0, 0xffffffffu, 0x00020000);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, dst + chunk(wave, i) * 64, 16, src.b_off[i], pair * src.b_step, 0, 0);
    }
    __device__ static __forceinline__ void issue(const P8Src &src, int wave, u32x4 *dst, int pair) {
#pragma unroll
        for (int i = 0; i < NB; ++i) issue1(src, wave, dst, pair, i);
    }
};

// This wave's LDS reads have returned.
__device__ __forceinline__ void wait_lds() {
    __builtin_amdgcn_s_waitcnt(0xc07f);                        // lgkmcnt(0)
    asm volatile("" ::: "memory");
}

// Order of a slab for the scheduler, in blocks of SIZE products: READS LDS reads (and VALU vector instructions) behind the first
// ones, loads behind the second half.
template <int BLOCKS, int SIZE, int READS, int VALU>
__device__ __forceinline__ void p8_spread_slab() {
#pragma unroll
    for (int m = 0; m < BLOCKS * SIZE; ++m) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (m % SIZE < READS) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        if (VALU > 0) __builtin_amdgcn_sched_group_barrier(0x002, VALU, 0);
        if (m % SIZE >= SIZE / 2) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
    }
}

// 16-bit weights.  Ring of DA + 1 slabs of weights and of PB pairs of slabs of tokens.  While slab s is multiplied, the operands of slab
// s + 1 are read into a second set of registers.  Slab s issues the loads of the weights of slab s + DA into the buffer that slab s - 1 has
// left; the last operands of pair p are read during slab 2 p, so slab 2 p + 1 issues, ahead of its weights, the tokens of pair p + PB
// into the buffer of pair p.  One wait and one barrier per slab publish slab s + 2.  The rings hold at most three pairs of slabs: what is
// fetched past the end of K has to land before LDS is given up, which in short products is much of their time, and a deeper ring brings
// nothing in long ones (panels of 128 x 192, five pairs -> three: 25 products of 5 to 12 us 4 % faster, K 2048 to 8192 level; with two
// pairs 128 x 64 takes 1.3 times as long).  128 x 64 then needs 80 KB, and two workgroups share a CU: grids of several rounds 1.2 times as fast.
// With one or two accumulator tiles in each direction a slab has too few products to spread its instructions under: the reads go in front, the loads
// between the two halves of the products (128 x 64 at K 512 5.9 -> 5.4 us with both changes, 4096 x 4096 at 64 tokens in eight slices 14.8 -> 14.3).
template <class T, int TB, int PR>
struct Panel8Loop16 : P8TokenPairs<TB, true> {
    using Tok = P8TokenPairs<TB, true>;
    static constexpr int A_SLAB = 512 * PR, RT = 2 * PR, TT = 2 * TB;       // granules of a slab of weights; row tiles, token blocks of a wave
    static constexpr size_t ring_bytes(int da, int pb) { return (size_t)((da + 1) * A_SLAB + pb * Tok::B_PAIR) * 16; }
    static constexpr int pairs(int pb) { return ring_bytes(2 * pb, pb + 1) <= kP8MostLds && pb < 3 ? pairs(pb + 1) : pb; }
    static constexpr int slabs(int da) { return da > 2 * PB - 2 && ring_bytes(da, PB) > kP8MostLds ? slabs(da - 1) : da; }
    static constexpr int PB = pairs(2), DA = slabs(2 * PB);
    static constexpr size_t lds_bytes = ring_bytes(DA, PB);
    static constexpr int B_AT = (DA + 1) * A_SLAB;
    static constexpr bool FEW = PR * TB <= 2;
    static_assert(lds_bytes <= kP8MostLds && DA >= 3 && DA >= 2 * PB - 2 && DA <= 2 * PB, "the rings have to fit, the waits below to hold");

    __device__ static __forceinline__ int tile(int wave, int i) { return PR * wave + i; }
    __device__ static __forceinline__ int pair(int) { return 0; }
    __device__ static __forceinline__ int scale_tile(int) { return 0; }

    __device__ static __forceinline__ void issue_a1(const P8Src &src, int wave, int slab, int buf, int i) {
        extern __shared__ u32x4 win[];
        __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)src.a, 16, 0xffffffffu, 1 << 23);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, win + buf * A_SLAB + (PR * wave + i) * 64, 16, 0, src.a_off[i] + slab * 1024, 0, 0);
    }

    // Slabs slab0 .. slab0 + nslab - 1; both numbers are even.  On return nothing is in flight and LDS is free once the workgroup
    // has met at a barrier.
    using Acc = P8Acc16<PR, TB>;
    template <int NS>
    __device__ static __forceinline__ void run(Acc &out, const P8Src &src, const ScaleRow (&)[NS], int slab0, int nslab,
                                               int wave, int lane) {
        extern __shared__ u32x4 win[];
        const int wr = wave & 3, wt = wave >> 2;
        const int a_idx = wr * RT * 64 + lane, b_idx[2] = {B_AT + Tok::operand16(src, 0, lane) + wt * TT * 128, B_AT + Tok::operand16(src, 1, lane) + wt * TT * 128};
        struct Frags {
            u32x4 a[RT], b[TT];
        } f0, f1;
        // read r of a slab: its row tiles first
        auto rd = [&](Frags &f, int abuf, int bbuf, int odd, int r) {
            if (r < RT) f.a[r] = win[abuf * A_SLAB + a_idx + r * 64];
            else f.b[r - RT] = win[bbuf * Tok::B_PAIR + b_idx[odd] + (r - RT) * 128];
        };
        constexpr int NR = RT + TT, NM = RT * TT, SIZE = NM % 8 ? 4 : 8, BLOCKS = NM / SIZE;
        // slabs past the end are fetched as copies of the last one and never multiplied, which keeps the count of loads in flight
        // the same in every trip
        const int last = slab0 + nslab - 1;
        auto issue_a = [&](int s, int buf, int i) { issue_a1(src, wave, min(slab0 + s, last), buf, i); };
        auto issue_b = [&](int s, int buf, int i) { Tok::issue1(src, wave, win + B_AT + buf * Tok::B_PAIR, min(slab0 + s, last) >> 1, i); };
        // the loads in front of slab 0 go out in the order in which the slabs before it would have issued them
#pragma unroll
        for (int v = DA > 2 * PB - 1 ? -DA : 1 - 2 * PB; v < 0; ++v) {
            if (v & 1 && v >= 1 - 2 * PB) {
#pragma unroll
                for (int i = 0; i < TB; ++i) issue_b(v - 1 + 2 * PB, (v - 1) / 2 + PB, i);
            }
#pragma unroll
            for (int i = 0; i < PR; ++i)
                if (v + DA >= 0) issue_a(v + DA, v + DA, i);
        }
        auto &acc = out.acc;
        out.zero();
        // Loads that may be in flight at the end of a slab s.  Behind the weights of slab s + 2 went out those of DA - 2 slabs and the
        // tokens of the odd slabs among them; behind the tokens of pair s / 2 + 1 (s even) the weights of 2 PB - 2 slabs and PB - 2
        // pairs of tokens.
        constexpr int ODD = (DA - 2) * PR + (DA - 1) / 2 * TB, EVEN_A = (DA - 2) * PR + (DA - 2) / 2 * TB;
        constexpr int EVEN_B = (2 * PB - 2) * PR + (PB - 2) * TB, EVEN = EVEN_A < EVEN_B ? EVEN_A : EVEN_B;
        constexpr int FIRST_B = (DA < 2 * PB - 1 ? DA : 2 * PB - 1) * PR + (PB - 1) * TB, FIRST = ODD < FIRST_B ? ODD : FIRST_B;
        wait_vmcnt_le<FIRST>();                                    // slabs 0 and 1, tokens of pair 0
        bare_barrier();
#pragma unroll
        for (int r = 0; r < NR; ++r) rd(f0, 0, 0, 0, r);
        int acur = 0, bcur = 0;                                    // buffers of slab s and of its pair
        auto trip = [&](int s, const Frags &now, Frags &next, auto odd_c) {
            constexpr int H = decltype(odd_c)::value, NL = PR + H * TB;
            const int anxt = acur == DA ? 0 : acur + 1, aprv = acur == 0 ? DA : acur - 1;
            const int bnxt = bcur == PB - 1 ? 0 : bcur + 1;
            auto load = [&](int l) {
                if (H && l < TB) issue_b(s - 1 + 2 * PB, bcur, l);
                else issue_a(s + DA, aprv, l - H * TB);
            };
            auto product = [&](int m) { acc[m / TT][m % TT] = T::mfma(now.a[m / TT], now.b[m % TT], acc[m / TT][m % TT]); };
            auto read = [&](int r) { rd(next, anxt, H ? bnxt : bcur, 1 - H, r); };
            if constexpr (FEW) {
#pragma unroll
                for (int m = 0; m < NM; ++m) product(m);
#pragma unroll
                for (int r = 0; r < NR; ++r) read(r);
#pragma unroll
                for (int l = 0; l < NL; ++l) load(l);
                __builtin_amdgcn_sched_group_barrier(0x100, NR, 0);                                   // LDS reads
                __builtin_amdgcn_sched_group_barrier(0x008, NM / 2, 0);                               // products
                __builtin_amdgcn_sched_group_barrier(0x020, NL, 0);                                   // loads
                __builtin_amdgcn_sched_group_barrier(0x008, NM / 2, 0);
            } else {
#pragma unroll
                for (int blk = 0; blk < BLOCKS; ++blk) {
#pragma unroll
                    for (int m = blk * SIZE; m < (blk + 1) * SIZE; ++m) product(m);
#pragma unroll
                    for (int r = 0; r < NR; ++r)
                        if (r * BLOCKS / NR == blk) read(r);
#pragma unroll
                    for (int l = 0; l < NL; ++l)
                        if ((l * BLOCKS + BLOCKS / 2) / NL == blk) load(l);
                }
                p8_spread_slab<BLOCKS, SIZE, (NR + BLOCKS - 1) / BLOCKS, 0>();
            }
            __builtin_amdgcn_sched_barrier(0);
            wait_vmcnt_le<H ? ODD : EVEN>();
            // the last operands of the pair have been read, not just asked for: its buffer is loaded over behind this barrier
            if (!H) wait_lds();
            bare_barrier();
            acur = anxt;
            if (H) bcur = bnxt;
        };
#pragma clang loop unroll(disable)
        for (int s = 0; s < nslab; s += 2) {
            trip(s, f0, f1, std::integral_constant<int, 0>());
            trip(s + 1, f1, f0, std::integral_constant<int, 1>());
        }
        __builtin_amdgcn_s_waitcnt(0);                             // nothing may still be writing LDS when the ring is given up
        mfma_settle();
    }
};

// Soft-FP8 weights of large panels.  The fp8 tiles (512 bytes) come through LDS as they are, and every wave widens the row tiles that it
// multiplies in registers, a slab ahead, between the products: each weight is widened by both token halves, four vector instructions a
// pair of them.  Widened once per workgroup and handed on through LDS as 16-bit tiles, as this loop once did, a slab moved 144 KiB
// through LDS, more than it passes while a slab is multiplied (28672 x 8192 at 1024 tokens 456 -> 411 us, in the 16 x 16 form).
// Ring of RP pairs of slabs, weights and tokens.  The last reads of pair p happen in slab 2 p; slab 2 p + 1 issues the tokens of pair
// p + RP into its place and slab 2 p + 2 the weights, so that one wait and one barrier per pair do, at the end of the even slab.
template <class T, int TB, int PR>
struct Panel8LoopFp8 : P8TokenPairs<TB, PR == 1> {
    using Tok = P8TokenPairs<TB, PR == 1>;
    static constexpr int RAW_PAIR = 512 * PR, SLOT = RAW_PAIR + Tok::B_PAIR, RT = 2 * PR, TT = 2 * TB;
    static constexpr size_t ring_bytes(int rp) { return (size_t)rp * SLOT * 16; }
    static constexpr int RP = 3;
    static constexpr size_t lds_bytes = ring_bytes(RP);
    static_assert(lds_bytes <= kP8MostLds, "the ring has to fit");

    __device__ static __forceinline__ int tile(int, int) { return 0; }
    __device__ static __forceinline__ int pair(int wave) { return PR == 2 ? wave : wave & 3; }
    __device__ static __forceinline__ int scale_tile(int wave) { return (wave & 3) * RT; }

    // the wave's load i < PR of a pair: two tiles of slab i (PR = 1: waves 0..3 fetch the first slab, 4..7 the second)
    __device__ static __forceinline__ void issue_a1(const P8Src &src, int wave, int pair, int buf, int i) {
        extern __shared__ u32x4 win[];
        __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)src.a, 0, 0xffffffffu, 0x00020000);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, win + buf * SLOT + (i * 8 + wave) * 64, 16, src.a_off[0],
                                                 (2 * pair + (PR == 2 ? i : wave >> 2)) * 512, 0, 0);
    }

    // As Panel8Loop16::run; srow[0]: block scales of the wave's rows, srow[1] (NS = 2): of its second half of row tiles
    // 256 rows: the 32 x 32 form, which leaves the vector unit more issue slots for the widening (panels of 256 x 256, 11008 x 4096 at 512
    // tokens 89 -> 76 us, 4096 x 14336 at 512 285 -> 244, 28672 x 8192 at 1024 411 -> 402).  128 rows, half as many weights a product: the
    // 16 x 16 form (8192 x 8192 at 2048 tokens in panels of 128 x 256: 32 x 32 275, 16 x 16 246).
    static constexpr bool M32 = PR == 2;
    using Acc = std::conditional_t<M32, P8Acc32<PR, TB>, P8Acc16<PR, TB>>;
    template <int NS>
    __device__ static __forceinline__ void run(Acc &out, const P8Src &src, const ScaleRow (&srow)[NS], int slab0, int nslab,
                                               int wave, int lane) {
        extern __shared__ u32x4 win[];
        const int wr = wave & 3, wt = wave >> 2;
        // operands of a slab: row tiles and blocks of 16 tokens, or (M32) those of row pair or block of 32 i / 2, k16 step i % 2
        const int a_idx = wr * RT * 64 + (M32 ? ((lane >> 4) & 1) * 64 + (lane >> 5) * 16 + (lane & 15) : lane);    // 8-byte units; second slab + 512 PR
        int b_idx[M32 ? 4 : 2];
#pragma unroll
        for (int h = 0; h < (M32 ? 4 : 2); ++h)
            b_idx[h] = RAW_PAIR + (M32 ? Tok::operand32(src, h, lane) : Tok::operand16(src, h, lane)) + wt * TT * 128;
        u32x4 a[2][RT], b[2][TT];
        u32x2 raw[RT];
        float sc[NS];
        auto rd_raw = [&](int buf, int odd, int i) {
            raw[i] = reinterpret_cast<const u32x2 *>(win + buf * SLOT)[a_idx + odd * 512 * PR + (M32 ? (i >> 1) * 128 + (i & 1) * 32 : i * 64)];
        };
        auto rd_b = [&](u32x4 (&f)[TT], int buf, int odd, int j) {
            f[j] = win[buf * SLOT + (M32 ? b_idx[2 * odd + (j & 1)] + (j >> 1) * 256 : b_idx[odd] + j * 128)];
        };
        auto widen = [&](u32x4 &o, int i) {
            const float s = sc[NS == 2 ? i / PR : 0];
            uint32_t x0, x1, x2, x3;
            fp8x4_to_bf16x4(raw[i][0], s, x0, x1);
            fp8x4_to_bf16x4(raw[i][1], s, x2, x3);
            o = u32x4{x0, x1, x2, x3};
        };
        const int pair0 = slab0 >> 1, npair = nslab >> 1, last = pair0 + npair - 1;
        auto scales = [&](int p) {
#pragma unroll
            for (int i = 0; i < NS; ++i) sc[i] = scale_at(srow[i], min(pair0 + p, last) >> 1);
        };
        // pairs past the end are fetched as copies of the last one and never multiplied
        auto issue_a = [&](int p, int buf, int i) { issue_a1(src, wave, min(pair0 + p, last), buf, i); };
        auto issue_b = [&](int p, int buf, int i) { Tok::issue1(src, wave, win + buf * SLOT + RAW_PAIR, min(pair0 + p, last), i); };
        constexpr int NM = M32 ? 2 * PR * TB : RT * TT, SIZE = M32 ? 4 : 8, BLOCKS = NM / SIZE;
        auto product = [&](const u32x4 (&x)[RT], const u32x4 (&y)[TT], int m) {
            if constexpr (M32) {
                const int hs = m / (PR * TB), pr = m / TB % PR, tb = m % TB;
                out.acc[pr][tb] = T::mfma32(x[2 * pr + hs], y[2 * tb + hs], out.acc[pr][tb]);
            } else {
                out.acc[m / TT][m % TT] = T::mfma(x[m / TT], y[m % TT], out.acc[m / TT][m % TT]);
            }
        };
#pragma unroll
        for (int p = 0; p < RP; ++p) {
#pragma unroll
            for (int i = 0; i < TB; ++i) issue_b(p, p, i);
#pragma unroll
            for (int i = 0; i < PR; ++i)
                if (p < RP - 1) issue_a(p, p, i);
        }
        out.zero();
        wait_vmcnt_le<(RP - 1) * TB + (RP - 2) * PR>();            // pair 0
        bare_barrier();
        scales(0);
#pragma unroll
        for (int i = 0; i < RT; ++i) rd_raw(0, 0, i);
#pragma unroll
        for (int j = 0; j < TT; ++j) rd_b(b[0], 0, 0, j);
#pragma unroll
        for (int i = 0; i < RT; ++i) widen(a[0][i], i);
        int cur = 0;                                               // buffer of pair p
#pragma clang loop unroll(disable)
        for (int p = 0; p < npair; ++p) {
            const int nxt = cur == RP - 1 ? 0 : cur + 1, prv = cur == 0 ? RP - 1 : cur - 1;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                // block blk multiplies, reads part of the next slab's operands and widens the tiles read before it
                if (h == 1) scales(p + 1);
                const int buf = h ? nxt : cur;
#pragma unroll
                for (int i = 0; i < RT; ++i) rd_raw(buf, 1 - h, i);
#pragma unroll
                for (int blk = 0; blk < BLOCKS; ++blk) {
#pragma unroll
                    for (int m = blk * SIZE; m < (blk + 1) * SIZE; ++m) product(a[h], b[h], m);
#pragma unroll
                    for (int i = 0; i < RT; ++i)
                        if (i * BLOCKS / RT == blk) widen(a[1 - h][i], i);
#pragma unroll
                    for (int j = 0; j < TT; ++j)
                        if (j * BLOCKS / TT == blk) rd_b(b[1 - h], buf, 1 - h, j);
                    if (h == 0) {
#pragma unroll
                        for (int i = 0; i < PR; ++i)
                            if ((i * BLOCKS + BLOCKS / 2) / PR == blk) issue_a(p + RP - 1, prv, i);
                    } else {
#pragma unroll
                        for (int i = 0; i < TB; ++i)
                            if ((i * BLOCKS + BLOCKS / 2) / TB == blk) issue_b(p + RP, cur, i);
                    }
                }
                p8_spread_slab<BLOCKS, SIZE, (RT + TT + BLOCKS - 1) / BLOCKS, (18 * RT + NM - 1) / NM>();
                __builtin_amdgcn_sched_barrier(0);
                if (h == 0) {
                    wait_vmcnt_le<(RP - 2) * (TB + PR)>();         // this wave's loads of pair p + 1 have landed
                    wait_lds();                                    // and it has all of pair p, which is loaded over behind this barrier
                    bare_barrier();
                }
            }
            cur = nxt;
        }
        __builtin_amdgcn_s_waitcnt(0);
        mfma_settle();
    }
};

}  // namespace mlk
