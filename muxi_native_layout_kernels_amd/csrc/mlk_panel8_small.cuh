// Main loops of the small eight-wave panels, 128 PR weight rows x 64 TB tokens with PR TB <= 4: what Panel8Loop
// (mlk_panel8.cuh) does for large ones, for panels that have few products to hide anything under.  Three things set the pace of a
// small panel, and each is met here.
//
// What a CU pulls.  Distinct weights come at 50 GB/s per CU at most (22 to 25 with all CUs at it: HBM), token rows that lie in L2 at
// 85 GB/s in whole 128-byte lines and half of that in pieces of 64 bytes.  Token rows are therefore fetched 64 k at a time:
// chunks of 8 tokens x 128 bytes, TB per wave for two k32 slabs.  Lane 8 r + j of a chunk's load fetches octet j ^ t of token
// t = r ^ (chunk & 1), so that the operand reads of 16 tokens meet 16 different bank groups.
//
// The round trip to memory.  The rings are as deep as LDS allows: with three slabs ahead a 128 x 64 panel ran at 0.34 us a slab
// whatever it multiplied.
//
// The round trip to LDS.  16-bit: the operands of a slab are read a whole slab ahead into a second set of registers.  Soft-FP8: a
// wave multiplies the rows it fetched the weights of, so that it widens its operands in registers and nothing but the tokens is
// shared.  Widened once per workgroup and handed on through LDS, as the large panels do, a slab took 0.28 us (128 x 64) to
// 0.42 us (256 x 64) without a single load in the loop: read, widen, write and a barrier one after the other.
#pragma once

#include "mlk_panel8.cuh"

namespace mlk {

// Chunks of 8 tokens x 64 k: which one load i of a wave brings, and this lane's part of it.
template <int TB>
struct P8TokenPairs {
    static constexpr int NB = TB, B_SLABS = 2, B_PAIR = 512 * TB;       // granules of a pair of slabs
    __device__ static __forceinline__ int chunk(int wave, int i) { return wave * TB + i; }
    __device__ static __forceinline__ int token_in_chunk(int wave, int i, int lane) { return (lane >> 3) ^ (chunk(wave, i) & 1); }
    __device__ static __forceinline__ int token(int wave, int i, int lane) { return chunk(wave, i) * 8 + token_in_chunk(wave, i, lane); }
    __device__ static __forceinline__ int octet(int wave, int i, int lane) { return (lane & 7) ^ token_in_chunk(wave, i, lane); }
    // granule of token lane % 32 of a block of 32 tokens, octet lane / 32; octet 2 h + lane / 32 is at ^ (2 h), block tb at + 256 tb
    __device__ static __forceinline__ int operand(int lane) {
        const int i = lane & 31, t = i & 7, c = i >> 3;
        return c * 64 + (t ^ (c & 1)) * 8 + ((lane >> 5) ^ t);
    }
    __device__ static __forceinline__ void issue(const P8Src &src, int wave, u32x4 *dst, int pair) {
        __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)src.b, 0, 0xffffffffu, 0x00020000);
#pragma unroll
        for (int i = 0; i < NB; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, dst + chunk(wave, i) * 64, 16, src.b_off[i], pair * src.b_step, 0, 0);
    }
};

// 16-bit weights.  Wave w = (token half w / 4, row quarter w % 4) as in Panel8Loop; ring of D + 1 slabs of weights and of
// D / 2 + 1 pairs of slabs of tokens.  Trip s issues the loads of the weights of slab s + D, even trips those of the tokens of slabs
// s + D and s + D + 1.
template <class T, int TB, int PR>
struct Panel8Small16 : P8TokenPairs<TB> {
    using Tok = P8TokenPairs<TB>;
    static constexpr int A_SLAB = 512 * PR;
    static constexpr size_t ring_bytes(int d) { return (size_t)((d + 1) * A_SLAB + (d / 2 + 1) * Tok::B_PAIR) * 16; }
    static constexpr int deepest(int d) { return ring_bytes(d + 2) <= kP8MostLds && d < 10 ? deepest(d + 2) : d; }
    static constexpr int D = deepest(4), PAIRS = D / 2 + 1;
    static constexpr size_t lds_bytes = ring_bytes(D);
    static constexpr int B_AT = (D + 1) * A_SLAB;
    static_assert(lds_bytes <= kP8MostLds, "the rings have to fit");

    __device__ static __forceinline__ int tile(int wave, int i) { return PR * wave + i; }
    __device__ static __forceinline__ int pair(int) { return 0; }

    __device__ static __forceinline__ void issue_a(const P8Src &src, int wave, int slab, int buf) {
        extern __shared__ u32x4 win[];
        __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)src.a, 16, 0xffffffffu, 1 << 23);
#pragma unroll
        for (int i = 0; i < PR; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, win + buf * A_SLAB + (PR * wave + i) * 64, 16, 0, src.a_off[i] + slab * 1024, 0, 0);
    }

    // acc[pr][tb] = rows of pair pr of this wave's quarter x tokens of block tb of its half, slabs slab0 .. slab0 + nslab - 1;
    // both numbers are even.  On return nothing is in flight and LDS is free once the workgroup has met at a barrier.
    __device__ static __forceinline__ void run(f32x16 (&acc)[PR][TB], const P8Src &src, const ScaleRow &, int slab0, int nslab, int wave,
                                               int lane) {
        extern __shared__ u32x4 win[];
        const int wr = wave & 3, wt = wave >> 2;
        const int a_idx = (wr * 2 * PR + ((lane >> 4) & 1)) * 64 + (lane >> 5) * 16 + (lane & 15);   // + 128 pr, + 32 second k16 step
        const int b_idx = Tok::operand(lane) + wt * TB * 256;
        struct Frags {
            u32x4 a[2][PR], b[2][TB];
        } f0, f1;
        auto rd = [&](Frags &f, int abuf, int bbuf, int odd) {
#pragma unroll
            for (int hs = 0; hs < 2; ++hs) {
#pragma unroll
                for (int pr = 0; pr < PR; ++pr) f.a[hs][pr] = win[abuf * A_SLAB + a_idx + 128 * pr + hs * 32];
#pragma unroll
                for (int tb = 0; tb < TB; ++tb) f.b[hs][tb] = win[B_AT + bbuf * Tok::B_PAIR + (b_idx ^ (4 * odd + 2 * hs)) + 256 * tb];
            }
        };
        // slabs past the end are fetched as copies of the last one and never multiplied, which keeps the count of loads in flight
        // the same in every trip
        const int last = slab0 + nslab - 1;
#pragma unroll
        for (int i = 0; i < D; ++i) {
            issue_a(src, wave, min(slab0 + i, last), i);
            if (i % 2 == 0) Tok::issue(src, wave, win + B_AT + i / 2 * Tok::B_PAIR, min(slab0 + i, last) >> 1);
        }
        zero_acc(acc);
        // All but this wave's loads of the youngest slabs have landed: D - 2 of weights and (D - 2) / 2 pairs of tokens were issued
        // behind those of slab s + 2, in odd trips (which issue weights only) and in even ones alike.
        constexpr int YOUNG = (D - 2) * PR + (D - 2) / 2 * TB;
        wait_vmcnt_le<YOUNG>();                                    // slabs 0 and 1
        bare_barrier();
        rd(f0, 0, 0, 0);
        int acur = 0, aprv = D, bcur = 0, bprv = PAIRS - 1;        // buffers of slab s and s - 1, of the pair of s and the one before
        auto trip = [&](int s, const Frags &now, Frags &next, auto odd_c) {
            constexpr int ODD = decltype(odd_c)::value;
            const int anxt = acur == D ? 0 : acur + 1, bnxt = bcur == PAIRS - 1 ? 0 : bcur + 1;
            issue_a(src, wave, min(slab0 + s + D, last), aprv);
            if constexpr (!ODD) Tok::issue(src, wave, win + B_AT + bprv * Tok::B_PAIR, min(slab0 + s + D, last) >> 1);
            rd(next, anxt, ODD ? bnxt : bcur, 1 - ODD);
#pragma unroll
            for (int hs = 0; hs < 2; ++hs)
#pragma unroll
                for (int tb = 0; tb < TB; ++tb)
#pragma unroll
                    for (int pr = 0; pr < PR; ++pr) acc[pr][tb] = T::mfma32(now.a[hs][pr], now.b[hs][tb], acc[pr][tb]);
            __builtin_amdgcn_sched_group_barrier(0x020, PR + (ODD ? 0 : TB), 0);                  // loads
            __builtin_amdgcn_sched_group_barrier(0x100, 2 * (PR + TB), 0);                        // LDS reads
            __builtin_amdgcn_sched_group_barrier(0x008, 2 * PR * TB, 0);                          // products
            __builtin_amdgcn_sched_barrier(0);
            wait_vmcnt_le<YOUNG>();                                // this wave's loads of slab s + 2 have landed
            bare_barrier();
            aprv = acur;
            acur = anxt;
            if (ODD) bprv = bcur, bcur = bnxt;
        };
        for (int s = 0; s < nslab; s += 2) {
            trip(s, f0, f1, std::integral_constant<int, 0>());
            trip(s + 1, f1, f0, std::integral_constant<int, 1>());
        }
        __builtin_amdgcn_s_waitcnt(0);                             // nothing may still be writing LDS when the ring is given up
        mfma_settle();
    }
};

// Soft-FP8 weights, in trips of two slabs (64 k).  A wave multiplies 32 rows, those of the two tiles it fetches itself into a part
// of LDS of its own, with all 64 TB tokens: PR = 2: the eight waves take the panel's 256 rows; PR = 1: waves w and w + 4 take the
// same 32 rows, w the even and w + 4 the odd slabs.  At the end the two waves of a row quarter exchange halves of their sums (PR = 1:
// and add them), so that every wave holds what Panel8Loop leaves in it.  Within a trip the token operands are read a k16 step
// ahead, the fp8 tiles two, and a step's weights are widened between the products of the step before.
template <class T, int TB, int PR>
struct Panel8SmallFp8 : P8TokenPairs<TB> {
    using Tok = P8TokenPairs<TB>;
    static constexpr int RAW_PAIR = 512 * PR, SLOT = RAW_PAIR + Tok::B_PAIR, TB2 = 2 * TB, NH = 2 * PR;     // k16 steps per trip
    static constexpr size_t ring_bytes(int d) { return (size_t)(d + 1) * SLOT * 16; }
    static constexpr int deepest(int d) { return ring_bytes(d + 1) <= kP8MostLds && d < 8 ? deepest(d + 1) : d; }
    static constexpr int D = deepest(3);                                 // pairs of slabs
    static constexpr size_t lds_bytes = ring_bytes(D);
    static_assert(lds_bytes <= kP8MostLds, "the rings have to fit");

    __device__ static __forceinline__ int tile(int, int) { return 0; }
    __device__ static __forceinline__ int pair(int wave) { return PR == 2 ? (wave & 3) * 2 + (wave >> 2) : wave & 3; }

    __device__ static __forceinline__ void issue(const P8Src &src, int wave, int pair, int buf) {
        extern __shared__ u32x4 win[];
        __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)src.a, 0, 0xffffffffu, 0x00020000);
#pragma unroll
        for (int i = 0; i < PR; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, win + buf * SLOT + (PR * wave + i) * 64, 16, src.a_off[0],
                                                     (2 * pair + (PR == 2 ? i : wave >> 2)) * 512, 0, 0);
        Tok::issue(src, wave, win + buf * SLOT + RAW_PAIR, pair);
    }

    __device__ static __forceinline__ void run(f32x16 (&acc)[PR][TB], const P8Src &src, const ScaleRow &srow, int slab0, int nslab,
                                               int wave, int lane) {
        extern __shared__ u32x4 win[];
        const int half = wave >> 2;
        const int a_idx = ((lane >> 4) & 1) * 64 + (lane >> 5) * 16 + (lane & 15);    // 8-byte units; second k16 step + 32, second slab + 128
        const int b_idx = RAW_PAIR + Tok::operand(lane);
        const int b_flip = PR == 1 ? 4 * half : 0;                                    // PR = 1: the slab of the pair that is this wave's
        u32x2 raw[2];                                                                 // tiles of the next two steps
        u32x4 op[2], b[2][TB2];
        f32x16 sum[TB2];
#pragma unroll
        for (int tb = 0; tb < TB2; ++tb)
#pragma unroll
            for (int e = 0; e < 16; ++e) sum[tb][e] = 0.f;
        auto rd_raw = [&](u32x2 &r, int buf, int h) {
            r = reinterpret_cast<const u32x2 *>(win + buf * SLOT + PR * wave * 64)[a_idx + (h >> 1) * 128 + (h & 1) * 32];
        };
        auto rd_b = [&](u32x4 (&f)[TB2], int buf, int h) {
#pragma unroll
            for (int tb = 0; tb < TB2; ++tb) f[tb] = win[buf * SLOT + (b_idx ^ (b_flip + 2 * h)) + 256 * tb];
        };
        auto widen = [&](u32x4 &o, const u32x2 &r, float sc) {
            uint32_t x0, x1, x2, x3;
            fp8x4_to_bf16x4(r[0], sc, x0, x1);
            fp8x4_to_bf16x4(r[1], sc, x2, x3);
            o = u32x4{x0, x1, x2, x3};
        };
        const int pair0 = slab0 >> 1, npair = nslab >> 1, last = pair0 + npair - 1;
#pragma unroll
        for (int i = 0; i < D; ++i) issue(src, wave, min(pair0 + i, last), i);
        constexpr int YOUNG = (D - 2) * (PR + TB);                 // loads issued behind those of pair p + 2
        wait_vmcnt_le<YOUNG>();                                    // pairs 0 and 1
        bare_barrier();
        float sc = scale_at(srow, pair0 >> 1);
        rd_raw(raw[0], 0, 0);
        rd_raw(raw[1], 0, 1);
        rd_b(b[0], 0, 0);
        widen(op[0], raw[0], sc);
        int cur = 0, prv = D;                                      // buffers of pair p and p - 1
        for (int p = 0; p < npair; ++p) {
            const int nxt = cur == D ? 0 : cur + 1;
            const float sc_next = scale_at(srow, min(pair0 + p + 1, last) >> 1);
#pragma unroll
            for (int h = 0; h < NH; ++h) {
                if (h + 1 < NH) rd_b(b[(h + 1) & 1], cur, h + 1);
                else rd_b(b[0], nxt, 0);
                if (h + 2 < NH) rd_raw(raw[h & 1], cur, h + 2);
                else rd_raw(raw[h & 1], nxt, h + 2 - NH);
                if (h == 0) issue(src, wave, min(pair0 + p + D, last), prv);
                widen(op[(h + 1) & 1], raw[(h + 1) & 1], h + 1 < NH ? sc : sc_next);
#pragma unroll
                for (int tb = 0; tb < TB2; ++tb) sum[tb] = T::mfma32(op[h & 1], b[h & 1][tb], sum[tb]);
                constexpr int PER = (18 + TB2 - 1) / TB2;          // conversion instructions per product
                __builtin_amdgcn_sched_group_barrier(0x100, TB2 + 1, 0);                          // LDS reads
                if (h == 0) __builtin_amdgcn_sched_group_barrier(0x020, PR + TB, 0);              // loads
#pragma unroll
                for (int m = 0; m < TB2; ++m) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, PER, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            wait_vmcnt_le<YOUNG>();                                // this wave's loads of pair p + 2 have landed
            bare_barrier();
            prv = cur;
            cur = nxt;
            sc = sc_next;
        }
        __builtin_amdgcn_s_waitcnt(0);
        mfma_settle();
        __syncthreads();                                           // LDS is free: the halves of the sums change hands through it
        f32x4 *mine = reinterpret_cast<f32x4 *>(win) + wave * TB * 256 + lane, *theirs = reinterpret_cast<f32x4 *>(win) + (wave ^ 4) * TB * 256 + lane;
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                f32x4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = half ? sum[tb][4 * q + e] : sum[TB + tb][4 * q + e];
                mine[(tb * 4 + q) * 64] = v;
            }
        __syncthreads();
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const f32x4 v = theirs[(tb * 4 + q) * 64];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float own = half ? sum[TB + tb][4 * q + e] : sum[tb][4 * q + e];
                    if constexpr (PR == 1) {
                        acc[0][tb][4 * q + e] = own + v[e];
                    } else {
                        acc[0][tb][4 * q + e] = half ? v[e] : own;
                        acc[1][tb][4 * q + e] = half ? own : v[e];
                    }
                }
            }
    }
};

// The loop of a panel shape.  (Soft-FP8 256 x 128 panels of grids of many rounds are level on both loops, 1.5 % behind to 4 % ahead on the
// small one; where they wait for weights it is 18 % ahead: expert layers, 8 experts at 300 tokens 490 -> 410 us.)
template <class T, bool FP8, int TB, int PR>
struct Panel8 {
    static constexpr bool SMALL = FP8 ? (PR == 2 ? TB <= 2 : TB <= 3) : PR * TB <= 4;
    using Loop = std::conditional_t<!SMALL, Panel8Loop<T, FP8, TB, PR>, std::conditional_t<FP8, Panel8SmallFp8<T, TB, PR>, Panel8Small16<T, TB, PR>>>;
};
// LDS of a kernel that runs the loops of TB = 1 .. tb.
template <bool FP8, int PR, int TB>
constexpr size_t p8_ring_bytes() {
    size_t most = Panel8<BF16, FP8, TB, PR>::Loop::lds_bytes;
    if constexpr (TB > 1) {
        const size_t other = p8_ring_bytes<FP8, PR, TB - 1>();
        if (other > most) most = other;
    }
    return most;
}

// A wave's token loads (row-major rows of `row_bytes`; token_of(slot): the row that a token slot of the panel reads).
template <class Loop, class TokenOf>
__device__ __forceinline__ void p8_token_rows(P8Src &src, uint32_t row_bytes, int wave, int lane, TokenOf token_of) {
    src.b_step = 64 * Loop::B_SLABS;
#pragma unroll
    for (int i = 0; i < Loop::NB; ++i)
        src.b_off[i] = (uint32_t)token_of(Loop::token(wave, i, lane)) * row_bytes + Loop::octet(wave, i, lane) * 16;
}
// The same from layout B ([K/32][m/16][4][16][8]).
template <class Loop, class TokenOf>
__device__ __forceinline__ void p8_token_native(P8Src &src, int m, int wave, int lane, TokenOf token_of) {
    src.b_step = (uint32_t)m * 64u * Loop::B_SLABS;
#pragma unroll
    for (int i = 0; i < Loop::NB; ++i) {
        const uint32_t tok = token_of(Loop::token(wave, i, lane)), oct = Loop::octet(wave, i, lane);
        src.b_off[i] = (oct >> 2) * ((uint32_t)m * 64u) + (tok >> 4) * 1024u + (oct & 3) * 256u + (tok & 15) * 16u;
    }
}

}  // namespace mlk
