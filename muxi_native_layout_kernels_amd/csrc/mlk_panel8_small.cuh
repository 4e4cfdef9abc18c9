// The soft-FP8 loop of the small eight-wave panels, 128 PR weight rows x 64 TB tokens (PR = 1 up to TB = 3, PR = 2 up to TB = 2), and the choice of a loop
// for a panel shape.  Three things set the pace of a small panel.
//
// What a CU pulls.  Distinct weights come at 50 GB/s per CU at most (22 to 25 with all CUs at it: HBM), token rows that lie in L2 at
// 85 GB/s in whole 128-byte lines and half of that in pieces of 64 bytes (hence P8TokenPairs).
//
// The round trip to memory.  The ring holds up to five pairs of slabs, four of them ahead: what is fetched past the end of K has to land before LDS
// is given up, which counts in short products (eight pairs ahead -> four, calls of 6 to 12 us: 128 x 64 3 % faster, 128 x 128 and 128 x 192
// 2 %; products of 12 to 50 us within 1 %, in slices of K 1 to 2 % faster).  128 x 64 then needs 80 KB, and two workgroups
// share a CU: grids of several rounds 1.25 times as fast.
//
// The round trip to LDS.  A wave multiplies the rows it fetched the weights of, so that it widens its operands in registers and nothing
// but the tokens is shared.  Widened once per workgroup and handed on through LDS, a slab took 0.28 us (128 x 64) to
// 0.42 us (256 x 64) without a single load in the loop: read, widen, write and a barrier one after the other.
#pragma once

#include "mlk_panel8.cuh"

namespace mlk {

// Soft-FP8 weights, in trips of two slabs (64 k).  A wave multiplies 32 rows, those of the two tiles it fetches itself into a part
// of LDS of its own, with all 64 TB tokens: PR = 2: the eight waves take the panel's 256 rows; PR = 1: waves w and w + 4 take the
// same 32 rows, w the even and w + 4 the odd slabs.  At the end the two waves of a row quarter exchange halves of their sums (PR = 1:
// and add them), so that every wave holds the sums of its row quarter and token half.  Within a trip the token operands are read a k16 step
// ahead, the fp8 tiles two, and a step's weights are widened between the products of the step before.
// v_mfma_f32_32x32x16 here: these panels are bound by the issue of vector instructions, and the 16 x 16 form takes twice as many (measured 9 to 12 %
// slower: 4096 x 14336, 200 tokens in panels of 256 x 128 153 -> 172 us, of 128 x 64 76 -> 83).
template <class T, int TB, int PR>
struct Panel8SmallFp8 : P8TokenPairs<TB, false> {
    using Tok = P8TokenPairs<TB, false>;
    static constexpr int RAW_PAIR = 512 * PR, SLOT = RAW_PAIR + Tok::B_PAIR, TB2 = 2 * TB, NH = 2 * PR;     // k16 steps per trip
    static constexpr size_t ring_bytes(int d) { return (size_t)(d + 1) * SLOT * 16; }
    static constexpr int deepest(int d) { return ring_bytes(d + 1) <= kP8MostLds && d < 4 ? deepest(d + 1) : d; }
    static constexpr int D = deepest(3);                                 // pairs of slabs
    static constexpr size_t lds_bytes = ring_bytes(D);
    static_assert(lds_bytes <= kP8MostLds, "the rings have to fit");

    __device__ static __forceinline__ int tile(int, int) { return 0; }
    __device__ static __forceinline__ int pair(int wave) { return PR == 2 ? (wave & 3) * 2 + (wave >> 2) : wave & 3; }
    __device__ static __forceinline__ int scale_tile(int wave) { return 2 * pair(wave); }

    __device__ static __forceinline__ void issue(const P8Src &src, int wave, int pair, int buf) {
        extern __shared__ u32x4 win[];
        __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)src.a, 0, 0xffffffffu, 0x00020000);
#pragma unroll
        for (int i = 0; i < PR; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, win + buf * SLOT + (PR * wave + i) * 64, 16, src.a_off[0],
                                                     (2 * pair + (PR == 2 ? i : wave >> 2)) * 512, 0, 0);
        Tok::issue(src, wave, win + buf * SLOT + RAW_PAIR, pair);
    }

    using Acc = P8Acc32<PR, TB>;
    template <int NS>
    __device__ static __forceinline__ void run(Acc &out, const P8Src &src, const ScaleRow (&srow)[NS], int slab0, int nslab, int wave,
                                               int lane) {
        extern __shared__ u32x4 win[];
        const int half = wave >> 2;
        const int a_idx = ((lane >> 4) & 1) * 64 + (lane >> 5) * 16 + (lane & 15);    // 8-byte units; second k16 step + 32, second slab + 128
        // step h is at b_idx ^ (h * b_step): those bits are clear in it.  (With the index of each step in a register of its own, expert layers of
        // 8 experts took 1 to 2 % longer at 264 to 352 tokens.)
        const int b_idx = RAW_PAIR + Tok::operand32(src, PR == 1 ? 2 * half : 0, lane);     // PR = 1: in the slab of the pair that is this wave's
        const int b_step = src.b_runs ? 32 : 2;
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
            for (int tb = 0; tb < TB2; ++tb) f[tb] = win[buf * SLOT + (b_idx ^ (h * b_step)) + 256 * tb];
        };
        // Where a trip's loads go out: in its second step; in the first, one behind each product (128 x 64, whose second step is its last:
        // 4 to 8 % slower there) or in front of the products (256 x 128, level).  All of them in front of the first step's products:
        // 128 x 128 1 to 2 % slower, 128 x 192 and 256 x 64 0.5 to 1 %, 128 x 64 1 %.
        constexpr bool SPREAD = PR * TB == 1;
        constexpr int LOADS = SPREAD || PR * TB == 4 ? 0 : 1;
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
        float sc = scale_at(srow[0], pair0 >> 1);
        rd_raw(raw[0], 0, 0);
        rd_raw(raw[1], 0, 1);
        rd_b(b[0], 0, 0);
        widen(op[0], raw[0], sc);
        int cur = 0, prv = D;                                      // buffers of pair p and p - 1
        for (int p = 0; p < npair; ++p) {
            const int nxt = cur == D ? 0 : cur + 1;
            const float sc_next = scale_at(srow[0], min(pair0 + p + 1, last) >> 1);
#pragma unroll
            for (int h = 0; h < NH; ++h) {
                if (h + 1 < NH) rd_b(b[(h + 1) & 1], cur, h + 1);
                else rd_b(b[0], nxt, 0);
                if (h + 2 < NH) rd_raw(raw[h & 1], cur, h + 2);
                else rd_raw(raw[h & 1], nxt, h + 2 - NH);
                if (h == LOADS) issue(src, wave, min(pair0 + p + D, last), prv);
                widen(op[(h + 1) & 1], raw[(h + 1) & 1], h + 1 < NH ? sc : sc_next);
#pragma unroll
                for (int tb = 0; tb < TB2; ++tb) sum[tb] = T::mfma32(op[h & 1], b[h & 1][tb], sum[tb]);
                constexpr int PER = (18 + TB2 - 1) / TB2;          // conversion instructions per product
                __builtin_amdgcn_sched_group_barrier(0x100, TB2 + 1, 0);                          // LDS reads
                if (h == LOADS && !SPREAD) __builtin_amdgcn_sched_group_barrier(0x020, PR + TB, 0);   // loads
#pragma unroll
                for (int m = 0; m < TB2; ++m) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, PER, 0);
                    if (h == LOADS && SPREAD) __builtin_amdgcn_sched_group_barrier(0x020, (PR + TB + TB2 - 1) / TB2, 0);
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
                        out.acc[0][tb][4 * q + e] = own + v[e];
                    } else {
                        out.acc[0][tb][4 * q + e] = half ? v[e] : own;
                        out.acc[1][tb][4 * q + e] = half ? own : v[e];
                    }
                }
            }
    }
};

// The loop of a panel shape.  (Soft-FP8 256 x 128 panels on the small loop and on the large one: 28672 x 8192 at 200 tokens 125 and 154 us, 4096 x
// 14336 at 400 153 and 200, 11008 x 4096 at 1000, several rounds, 116 and 133.)
template <class T, bool FP8, int TB, int PR>
struct Panel8 {
    static constexpr bool SMALL = PR == 2 ? TB <= 2 : TB <= 3;
    using Loop = std::conditional_t<!FP8, Panel8Loop16<T, TB, PR>, std::conditional_t<SMALL, Panel8SmallFp8<T, TB, PR>, Panel8LoopFp8<T, TB, PR>>>;
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
    src.b_step = 128;
    src.b_runs = false;
#pragma unroll
    for (int i = 0; i < Loop::NB; ++i)
        src.b_off[i] = (uint32_t)token_of(Loop::token(wave, i, lane)) * row_bytes + Loop::octet(wave, i, lane) * 16;
}
// The same from layout B ([K/32][m/16][4][16][8]).
template <class Loop, class TokenOf>
__device__ __forceinline__ void p8_token_native(P8Src &src, int m, int wave, int lane, TokenOf token_of) {
    src.b_step = (uint32_t)m * 128u;
    src.b_runs = true;
#pragma unroll
    for (int i = 0; i < Loop::NB; ++i) {
        const int chunk = Loop::chunk(wave, i);
        src.b_off[i] = (uint32_t)(chunk & 1) * ((uint32_t)m * 64u) + ((uint32_t)token_of((chunk >> 1) * 16) >> 4) * 1024u + lane * 16u;
    }
}

}  // namespace mlk
