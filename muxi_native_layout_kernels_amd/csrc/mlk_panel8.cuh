// Main loop of the eight-wave panels: 256 weight rows x 64 TB tokens (TB = 1..4), both operands through LDS, fetched
// with loads that write LDS directly, v_mfma_f32_32x32x16.
//
// A wave that issues v_mfma_f32_32x32x16 back to back loses matrix-core time with every other instruction it has to
// issue in between (measured: about 20 cycles per LDS read, 24 per load); with two waves per SIMD the instructions
// of one wave go out under the products of the other.  That needs both waves of a SIMD inside 256 registers each,
// so nothing is staged through registers here: a k32 slab of the panel (16 weight tiles of 16 rows x 32 k, 1 KiB
// each, as they lie in layout A; 4 TB chunks of 16 tokens x 32 k) is copied into LDS by buffer loads with the LDS
// bit: per wave two weight tiles, addressed by the thread id alone (the descriptor adds 16 bytes per lane, no
// address register), and its token chunks with a per-lane offset (lane 4 t + j fetches octet j ^ (t / 4) of token t, so
// that four lanes cover 64 consecutive bytes of a token row and the operand reads below meet no bank twice).
// Wave w = (token half w / 4, row quarter w % 4) multiplies 64 rows x 32 TB tokens: per k16 step two weight operands (two
// vertically adjacent tiles read as one 32-row operand: lane 32 g + i takes row i % 16 of tile i / 16, octet g) and TB
// token operands feed 2 TB products.
//
// Ring of four slabs (128 KiB).  While slab s is multiplied, slab s + 1 is complete and published, slab s + 2 is landing
// and the loads of slab s + 3 go out into the buffer that slab s - 1 has left; one wait (this wave's loads of slab
// s + 2) and one barrier per slab publish slab s + 2 and retire slab s.  The operands of the first step of slab s + 1
// are read before that barrier, so no wave stands idle behind it.  The barrier is the bare instruction: the fence that
// comes with __syncthreads() would wait for every load in flight.
//
// Soft-FP8 weights: the fp8 tiles (512 bytes) land in a small ring of their own (three slabs of 8 KiB behind the four
// bf16 slabs: 152 KiB in all); every wave widens the two tiles it fetched itself, two slabs ahead of their use, lane by
// lane (8 bytes in, 16 bytes out at the same lane's place: the tile order does not change) into the bf16 slab, so that
// each weight is widened once per workgroup and the multiplying loop is the 16-bit one.
#pragma once

#include "mlk_panel_lds.cuh"

namespace mlk {

constexpr int kP8Slab = 2048;                                  // 16-byte granules of a slab: 1024 of weights, 1024 of tokens
constexpr size_t kP8RingBytes = (size_t)4 * kP8Slab * 16;
constexpr int kP8RawSlab = 512;                                // granules of a slab of fp8 tiles
constexpr size_t kP8Fp8LdsBytes = (size_t)(4 * kP8Slab + 3 * kP8RawSlab) * 16;

// Token chunks (16 tokens each) a wave fetches per slab, and which ones.  With three and one blocks per token half there
// are fewer chunks than wave slots; the spare slots fetch a chunk a second time (the same bytes to the same place), which
// keeps the count of loads in flight equal in all waves.
template <int TB>
__host__ __device__ constexpr int p8_chunk_loads() {
    return TB >= 3 ? 2 : 1;
}
template <int TB>
__device__ __forceinline__ int p8_chunk(int wave, int i) {
    if (TB == 4) return 2 * wave + i;
    if (TB == 3) return i == 0 ? wave : (wave < 4 ? wave + 8 : wave);
    if (TB == 2) return wave;
    return wave & 3;
}

// Where a wave's loads come from.
struct P8Src {
    const uint8_t *a;      // workgroup-uniform base of the weight tiles
    uint32_t a_off[2];     // 16-bit: wave-uniform byte offsets of the wave's two tiles at k = 0; fp8: [0] = per-lane byte
                           // offset (lanes 0..31 the first tile, 32..63 the second, 16 bytes each)
    const uint16_t *b;     // base of the token rows
    uint32_t b_off[2];     // per-lane byte offsets of this lane's 16 bytes of the wave's chunks at k = 0
};
// Byte offset of this lane's 16 bytes of a chunk from the row that token lane / 4 of the chunk reads.
__device__ __forceinline__ uint32_t p8_lane_octet(int lane) {
    const int t = lane >> 2;
    return (uint32_t)((lane & 3) ^ ((t >> 2) & 3)) * 16;
}

template <class T, bool FP8, int TB>
struct Panel8Loop {
    static constexpr int PR = 2, RING = 4, NB = p8_chunk_loads<TB>(), NA = FP8 ? 1 : 2;

    __device__ static __forceinline__ void issue_b(const P8Src &src, int wave, int slab, int buf) {
        extern __shared__ u32x4 win[];
        __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)src.b, 0, 0xffffffffu, 0x00020000);
#pragma unroll
        for (int i = 0; i < NB; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, win + buf * kP8Slab + 1024 + p8_chunk<TB>(wave, i) * 64, 16, src.b_off[i],
                                                     slab * 64, 0, 0);
    }
    __device__ static __forceinline__ void issue_a(const P8Src &src, int wave, int slab, int buf) {
        extern __shared__ u32x4 win[];
        if constexpr (FP8) {
            __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)src.a, 0, 0xffffffffu, 0x00020000);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, win + 4 * kP8Slab + buf * kP8RawSlab + 2 * wave * 32, 16, src.a_off[0],
                                                     slab * 512, 0, 0);
        } else {
            __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)src.a, 16, 0xffffffffu, 1 << 23);
#pragma unroll
            for (int i = 0; i < 2; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, win + buf * kP8Slab + (2 * wave + i) * 64, 16, 0,
                                                         src.a_off[i] + slab * 1024, 0, 0);
        }
    }

    // acc[pr][tb] += rows of pair pr of this wave's quarter x tokens of block tb of its half, slabs slab0 .. slab0 + nslab - 1.
    // On return nothing is in flight and the LDS ring is free once the workgroup has met at a barrier.
    __device__ static __forceinline__ void run(f32x16 (&acc)[PR][TB], const P8Src &src, const ScaleRow &srow, int slab0, int nslab,
                                               int wave, int lane) {
        extern __shared__ u32x4 win[];
        const int wr = wave & 3, wt = wave >> 2;
        // operand reads (granules inside a slab, first k16 step; the second step is + 32 for weights, ^ 2 for tokens)
        const int g = lane >> 5, t16 = lane & 15, hi = (lane >> 4) & 1;
        const int a_idx = (wr * 4 + hi) * 64 + g * 16 + t16;                                         // + 128 pr
        const int b_idx = 1024 + (wt * 2 * TB + hi) * 64 + 4 * t16 + (g ^ ((t16 >> 2) & 3));         // + 128 tb
        u32x4 a0[PR], a1[PR], b0[TB], b1[TB];
        auto rd = [&](u32x4 (&a)[PR], u32x4 (&b)[TB], int buf, int hs) {
            const u32x4 *s = win + buf * kP8Slab;
#pragma unroll
            for (int pr = 0; pr < PR; ++pr) a[pr] = s[a_idx + 128 * pr + hs * 32];
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) b[tb] = s[(b_idx ^ (hs * 2)) + 128 * tb];
        };
        auto mm = [&](const u32x4 (&a)[PR], const u32x4 (&b)[TB]) {
#pragma unroll
            for (int tb = 0; tb < TB; ++tb)
#pragma unroll
                for (int pr = 0; pr < PR; ++pr) acc[pr][tb] = T::mfma32(a[pr], b[tb], acc[pr][tb]);
        };
        // slabs past the end are fetched as copies of the last slab and never multiplied, which keeps the count of loads
        // in flight the same in every trip
        const int last = slab0 + nslab - 1;
        if constexpr (!FP8) {
#pragma unroll
            for (int i = 0; i < RING - 1; ++i) {
                issue_a(src, wave, min(slab0 + i, last), i);
                issue_b(src, wave, min(slab0 + i, last), i);
            }
            wait_vmcnt_le<(NA + NB) * (RING - 3)>();               // slabs 0 and 1 of this wave have landed
            bare_barrier();
            rd(a0, b0, 0, 0);
            int cur = 0;                                           // ring buffer of slab s
            for (int s = 0; s < nslab; ++s) {
                const int nxt = (cur + 1) & 3, prv = (cur + 3) & 3;
                rd(a1, b1, cur, 1);
                issue_a(src, wave, min(slab0 + s + RING - 1, last), prv);
                issue_b(src, wave, min(slab0 + s + RING - 1, last), prv);
                mm(a0, b0);
                spread_half_step<2 * TB, PR + TB, NA + NB>();
                rd(a0, b0, nxt, 0);
                mm(a1, b1);
                spread_half_step<2 * TB, PR + TB, 0>();
                wait_vmcnt_le<(NA + NB) * (RING - 3)>();           // this wave's loads of slab s + 2 have landed
                bare_barrier();
                cur = nxt;
            }
        } else {
            // widen this wave's two tiles of slab `slab` (counted from k = 0) from raw buffer rb into bf16 slab buffer `buf`
            auto widen = [&](int slab, int rb, int buf) {
                const float sc = scale_at(srow, slab >> 2);
                const u32x2 *raw = reinterpret_cast<const u32x2 *>(win + 4 * kP8Slab + rb * kP8RawSlab + 2 * wave * 32);
                u32x4 *dst = win + buf * kP8Slab + 2 * wave * 64;
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const u32x2 f = raw[i * 64 + lane];
                    uint32_t x0, x1, x2, x3;
                    fp8x4_to_bf16x4(f[0], sc, x0, x1);
                    fp8x4_to_bf16x4(f[1], sc, x2, x3);
                    dst[i * 64 + lane] = u32x4{x0, x1, x2, x3};
                }
            };
            // Order of this wave's loads: chunks(0) raw(0) chunks(1) raw(1) chunks(2) raw(2) | raw(3) | then per trip s:
            // chunks(s + 3) raw(s + 4).
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                issue_b(src, wave, min(slab0 + i, last), i);
                issue_a(src, wave, min(slab0 + i, last), i);
            }
            wait_vmcnt_le<NB + 1>();                               // chunks and tiles of slabs 0 and 1 have landed
            widen(min(slab0, last), 0, 0);
            widen(min(slab0 + 1, last), 1, 1);
            issue_a(src, wave, min(slab0 + 3, last), 0);           // raw(3) into the raw buffer that slab 0 has left
            if constexpr (TB > 1) wait_vmcnt_le<1>();              // the tiles of slab 2
            __builtin_amdgcn_s_waitcnt(0xc07f);                    // lgkmcnt(0): the widened tiles are written
            bare_barrier();
            rd(a0, b0, 0, 0);
            int cur = 0, rcur = 0;                                 // ring buffer of slab s, raw buffer of slab s
            for (int s = 0; s < nslab; ++s) {
                const int nxt = (cur + 1) & 3, nx2 = (cur + 2) & 3, prv = (cur + 3) & 3;
                const int r1 = rcur == 2 ? 0 : rcur + 1, r2 = rcur == 0 ? 2 : rcur - 1;  // raw buffers of slabs s + 1 (= s + 4), s + 2
                auto issue = [&]() {
                    issue_b(src, wave, min(slab0 + s + 3, last), prv);
                    issue_a(src, wave, min(slab0 + s + 4, last), r1);
                };
                // With 64 token columns a slab has four products to hide anything under and latency sets the pace: the loads go
                // out first, the operands are read in front of the products, and the tiles of slab s + 2 are waited for only
                // here, a trip later than with more columns (the loads of two trips may be in flight; in the first one raw(3),
                // which went out alone, and this trip's).  256 experts top-8, I 256, at 300 tokens: 487 -> 467 us.
                if constexpr (TB == 1) {
                    issue();
                    if (s == 0) wait_vmcnt_le<NB + 2>();
                    else wait_vmcnt_le<2 * (NB + 1)>();
                }
                // The fp8 tiles of slab s + 2 are read first, widened between the products of the first half step and written
                // after them.  From 128 columns on the loads go out behind the LDS reads, under the products (see
                // spread_half_step); issued in front of them, right behind the barrier, every wave stood still for them:
                // 28672 x 8192 at 1024 tokens 454 -> 444 us.
                const float sc = scale_at(srow, min(slab0 + s + 2, last) >> 2);
                const u32x2 *raw = reinterpret_cast<const u32x2 *>(win + 4 * kP8Slab + r2 * kP8RawSlab + 2 * wave * 32);
                const u32x2 f0 = raw[lane], f1 = raw[64 + lane];
                rd(a1, b1, cur, 1);
                if constexpr (TB > 1) issue();
                u32x4 w0, w1;
                {
                    uint32_t x0, x1, x2, x3;
                    fp8x4_to_bf16x4(f0[0], sc, x0, x1);
                    fp8x4_to_bf16x4(f0[1], sc, x2, x3);
                    w0 = u32x4{x0, x1, x2, x3};
                    fp8x4_to_bf16x4(f1[0], sc, x0, x1);
                    fp8x4_to_bf16x4(f1[1], sc, x2, x3);
                    w1 = u32x4{x0, x1, x2, x3};
                }
                mm(a0, b0);
                {
                    u32x4 *dst = win + nx2 * kP8Slab + 2 * wave * 64;
                    dst[lane] = w0;
                    dst[64 + lane] = w1;
                }
                if constexpr (TB >= 2) {
                    constexpr int NM = 2 * TB, NR = 2 + PR + TB, PER = (36 + NM - 3) / (NM - 2);   // conversion instructions per gap
                    constexpr int S0 = (NR + 1) / 2, LPER = (NB + 1 + NM - S0 - 1) / (NM - S0);    // first gap with loads, loads per gap
                    __builtin_amdgcn_sched_group_barrier(0x006, 24, 0);                            // addresses
#pragma unroll
                    for (int m = 0; m < NM; ++m) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        if (2 * m + 1 < NR) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                        else if (2 * m < NR) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                        if (m >= 2) __builtin_amdgcn_sched_group_barrier(0x002, PER, 0);
                        if (m >= S0 && (m - S0) * LPER < NB + 1) __builtin_amdgcn_sched_group_barrier(0x020, LPER, 0);
                    }
                    __builtin_amdgcn_sched_group_barrier(0x200, 2, 0);                             // the two LDS writes
                } else {
                    __builtin_amdgcn_sched_group_barrier(0x100, 2 + PR + TB, 0);                   // the LDS reads
                }
                __builtin_amdgcn_sched_barrier(0);
                rd(a0, b0, nxt, 0);
                mm(a1, b1);
                if constexpr (TB > 1) spread_half_step<2 * TB, PR + TB, 0>();
                else __builtin_amdgcn_sched_barrier(0);
                // this wave's chunks of slab s + 2 have landed, and (but for 64 token columns) its tiles of slab s + 3
                wait_vmcnt_le<TB == 1 ? NB + 2 : NB + 1>();
                __builtin_amdgcn_s_waitcnt(0xc07f);                // and its widened tiles are written
                bare_barrier();
                cur = nxt;
                rcur = r1;
            }
        }
        __builtin_amdgcn_s_waitcnt(0);                             // nothing may still be writing LDS when the ring is given up
        mfma_settle();
    }
};

template <int PR, int TB>
__device__ __forceinline__ void zero_acc(f32x16 (&acc)[PR][TB]) {
#pragma unroll
    for (int pr = 0; pr < PR; ++pr)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[pr][tb][e] = 0.f;
}

}  // namespace mlk
