// Main loops of the eight-wave panels: 128 PR weight rows x 64 TB tokens (PR = 1, 2; TB = 1..4), both operands through LDS,
// fetched with loads that write LDS directly, v_mfma_f32_32x32x16.  Panel8Loop is for the large panels (256 x 192 and 256 x 256,
// soft-FP8 also 128 x 256), the two of mlk_panel8_small.cuh for the others; Panel8<..>::Loop picks.
//
// A wave that issues v_mfma_f32_32x32x16 back to back loses matrix-core time with every other instruction it has to
// issue in between (measured: about 20 cycles per LDS read, 24 per load); with two waves per SIMD the instructions
// of one wave go out under the products of the other.  That needs both waves of a SIMD inside 256 registers each,
// so nothing is staged through registers here: a k32 slab of the panel (8 PR weight tiles of 16 rows x 32 k, 1 KiB
// each, as they lie in layout A; 4 TB chunks of 16 tokens x 32 k) is copied into LDS by buffer loads with the LDS
// bit: per wave PR weight tiles, addressed by the thread id alone (the descriptor adds 16 bytes per lane, no
// address register), and its token chunks with a per-lane offset (lane 4 t + j fetches octet j ^ (t / 4) of token t, so
// that four lanes cover 64 consecutive bytes of a token row and the operand reads below meet no bank twice; a chunk of
// layout-B activations is one run of 1 KiB, of which the lane takes the granule of the same octet and token).
// Wave w = (token half w / 4, row quarter w % 4) multiplies 32 PR rows x 32 TB tokens: per k16 step PR weight operands (two
// vertically adjacent tiles read as one 32-row operand: lane 32 g + i takes row i % 16 of tile i / 16, octet g) and TB
// token operands feed PR TB products.
//
// Ring of four slabs (128 KiB for 256 x 256).  While slab s is multiplied, slab s + 1 is complete and published, slab s + 2 is landing
// and the loads of slab s + 3 go out into the buffer that slab s - 1 has left; one wait (this wave's loads of slab
// s + 2) and one barrier per slab publish slab s + 2 and retire slab s.  The operands of the first step of slab s + 1
// are read before that barrier, so no wave stands idle behind it.  The barrier is the bare instruction: the fence that
// comes with __syncthreads() would wait for every load in flight.
//
// Soft-FP8 weights: the fp8 tiles (512 bytes) land in a small ring of their own (three slabs of 8 KiB behind the four
// bf16 slabs: 152 KiB in all); every wave widens the PR tiles it fetched itself, two slabs ahead of their use, lane by
// lane (8 bytes in, 16 bytes out at the same lane's place: the tile order does not change) into the bf16 slab, so that
// each weight is widened once per workgroup and the multiplying loop is the 16-bit one.  A load moves 1 KiB, two tiles: with
// PR = 1 two neighbouring waves fetch the same two tiles, each to a place of its own, and widen one each.
#pragma once

#include "mlk_panel_lds.cuh"

namespace mlk {

constexpr size_t kP8MostLds = 152 * 1024;                      // of a ring

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

// Where a wave's loads come from.  A loop says which weight tiles and which tokens a wave fetches: tile(wave, i) for i < PR (16-bit),
// pair(wave): the two tiles 2 pair, 2 pair + 1 (soft-FP8); token(wave, i, lane) and octet(wave, i, lane), the 8 k of a group of
// B_SLABS slabs, for i < NB.
struct P8Src {
    const uint8_t *a;      // workgroup-uniform base of the weight tiles
    uint32_t a_off[2];     // 16-bit: wave-uniform byte offsets of the wave's PR tiles at k = 0; fp8: [0] = per-lane byte
                           // offset (lanes 0..31 the first tile, 32..63 the second, 16 bytes each)
    const uint16_t *b;     // base of the token rows
    uint32_t b_off[4];     // per-lane byte offsets of this lane's 16 bytes of the wave's chunks at k = 0
    uint32_t b_step;       // bytes from one group of B_SLABS slabs to the next: of a token row, or of all tokens in layout B
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

template <class T, bool FP8, int TB, int PR>
struct Panel8Loop {
    static_assert(PR * TB >= 4, "smaller panels have too few products per half step to hide anything under");
    static constexpr int RING = 4, NB = p8_chunk_loads<TB>(), NA = FP8 ? 1 : PR, B_SLABS = 1;
    // granules: a slab, its first token chunk, a slab of fp8 tiles
    static constexpr int SLAB = 512 * PR + 256 * TB, BOFF = 512 * PR, RAW_SLAB = 512;
    static constexpr size_t lds_bytes = (size_t)(RING * SLAB + (FP8 ? 3 * RAW_SLAB : 0)) * 16;

    __device__ static __forceinline__ int tile(int wave, int i) { return PR * wave + i; }
    __device__ static __forceinline__ int pair(int wave) { return PR == 2 ? wave : wave >> 1; }
    __device__ static __forceinline__ int token(int wave, int i, int lane) { return p8_chunk<TB>(wave, i) * 16 + (lane >> 2); }
    __device__ static __forceinline__ int octet(int wave, int i, int lane) { return (lane & 3) ^ ((lane >> 4) & 3); }

    __device__ static __forceinline__ void issue_b(const P8Src &src, int wave, int slab, int buf) {
        extern __shared__ u32x4 win[];
        __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)src.b, 0, 0xffffffffu, 0x00020000);
#pragma unroll
        for (int i = 0; i < NB; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, win + buf * SLAB + BOFF + p8_chunk<TB>(wave, i) * 64, 16, src.b_off[i],
                                                     slab * src.b_step, 0, 0);
    }
    __device__ static __forceinline__ void issue_a(const P8Src &src, int wave, int slab, int buf) {
        extern __shared__ u32x4 win[];
        if constexpr (FP8) {
            __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)src.a, 0, 0xffffffffu, 0x00020000);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, win + RING * SLAB + buf * RAW_SLAB + wave * 64, 16, src.a_off[0],
                                                     slab * 512, 0, 0);
        } else {
            __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)src.a, 16, 0xffffffffu, 1 << 23);
#pragma unroll
            for (int i = 0; i < PR; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, win + buf * SLAB + (PR * wave + i) * 64, 16, 0,
                                                         src.a_off[i] + slab * 1024, 0, 0);
        }
    }

    // acc[pr][tb] = rows of pair pr of this wave's quarter x tokens of block tb of its half, slabs slab0 .. slab0 + nslab - 1.
    // On return nothing is in flight and the LDS ring is free once the workgroup has met at a barrier.
    __device__ static __forceinline__ void run(f32x16 (&acc)[PR][TB], const P8Src &src, const ScaleRow &srow, int slab0, int nslab,
                                               int wave, int lane) {
        extern __shared__ u32x4 win[];
        const int wr = wave & 3, wt = wave >> 2;
        // operand reads (granules inside a slab, first k16 step; the second step is + 32 for weights, ^ 2 for tokens)
        const int g = lane >> 5, t16 = lane & 15, hi = (lane >> 4) & 1;
        const int a_idx = (wr * 2 * PR + hi) * 64 + g * 16 + t16;                                    // + 128 pr
        const int b_idx = BOFF + (wt * 2 * TB + hi) * 64 + 4 * t16 + (g ^ ((t16 >> 2) & 3));         // + 128 tb
        u32x4 a0[PR], a1[PR], b0[TB], b1[TB];
        auto rd = [&](u32x4 (&a)[PR], u32x4 (&b)[TB], int buf, int hs) {
            const u32x4 *s = win + buf * SLAB;
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
        zero_acc(acc);
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
                spread_half_step<PR * TB, PR + TB, NA + NB>();
                rd(a0, b0, nxt, 0);
                mm(a1, b1);
                spread_half_step<PR * TB, PR + TB, 0>();
                wait_vmcnt_le<(NA + NB) * (RING - 3)>();           // this wave's loads of slab s + 2 have landed
                bare_barrier();
                cur = nxt;
            }
        } else {
            // widen this wave's tiles of slab `slab` (counted from k = 0) from raw buffer rb into bf16 slab buffer `buf`
            const int mine = PR == 2 ? 0 : (wave & 1) * 64;        // of the two tiles that came with this wave's loads
            auto raw_tiles = [&](u32x2 (&f)[PR], int rb) {
#pragma unroll
                for (int i = 0; i < PR; ++i)
                    f[i] = reinterpret_cast<const u32x2 *>(win + RING * SLAB + rb * RAW_SLAB + wave * 64)[mine + i * 64 + lane];
            };
            auto widen = [&](u32x4 (&w)[PR], const u32x2 (&f)[PR], float sc) {
#pragma unroll
                for (int i = 0; i < PR; ++i) {
                    uint32_t x0, x1, x2, x3;
                    fp8x4_to_bf16x4(f[i][0], sc, x0, x1);
                    fp8x4_to_bf16x4(f[i][1], sc, x2, x3);
                    w[i] = u32x4{x0, x1, x2, x3};
                }
            };
            auto put = [&](const u32x4 (&w)[PR], int buf) {
#pragma unroll
                for (int i = 0; i < PR; ++i) win[buf * SLAB + (PR * wave + i) * 64 + lane] = w[i];
            };
            u32x2 f[PR];
            u32x4 w[PR];
            // Order of this wave's loads: chunks(0) raw(0) chunks(1) raw(1) chunks(2) raw(2) | raw(3) | then per trip s:
            // chunks(s + 3) raw(s + 4).
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                issue_b(src, wave, min(slab0 + i, last), i);
                issue_a(src, wave, min(slab0 + i, last), i);
            }
            wait_vmcnt_le<NB + 1>();                               // chunks and tiles of slabs 0 and 1 have landed
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                raw_tiles(f, i);
                widen(w, f, scale_at(srow, min(slab0 + i, last) >> 2));
                put(w, i);
            }
            // raw(3) goes where the tiles of slab 0 were: only once they have been read (a load that finds its lines in the cache of
            // the CU can be ahead of an LDS read issued before it)
            __builtin_amdgcn_s_waitcnt(0xc07f);                    // lgkmcnt(0)
            asm volatile("" ::: "memory");
            issue_a(src, wave, min(slab0 + 3, last), 0);
            wait_vmcnt_le<1>();                                    // the tiles of slab 2
            __builtin_amdgcn_s_waitcnt(0xc07f);                    // lgkmcnt(0): the widened tiles are written
            bare_barrier();
            rd(a0, b0, 0, 0);
            int cur = 0, rcur = 0;                                 // ring buffer of slab s, raw buffer of slab s
            for (int s = 0; s < nslab; ++s) {
                const int nxt = (cur + 1) & 3, nx2 = (cur + 2) & 3, prv = (cur + 3) & 3;
                const int r1 = rcur == 2 ? 0 : rcur + 1, r2 = rcur == 0 ? 2 : rcur - 1;  // raw buffers of slabs s + 1 (= s + 4), s + 2
                // The fp8 tiles of slab s + 2 are read first, widened between the products of the first half step and written
                // after them.  From 128 columns on the loads go out behind the LDS reads, under the products (see
                // spread_half_step); issued in front of them, right behind the barrier, every wave stood still for them:
                // 28672 x 8192 at 1024 tokens 454 -> 444 us.
                const float sc = scale_at(srow, min(slab0 + s + 2, last) >> 2);
                raw_tiles(f, r2);
                rd(a1, b1, cur, 1);
                issue_b(src, wave, min(slab0 + s + 3, last), prv);
                issue_a(src, wave, min(slab0 + s + 4, last), r1);
                widen(w, f, sc);
                mm(a0, b0);
                put(w, nx2);
                {
                    constexpr int NM = PR * TB, NR = PR + PR + TB, PER = (18 * PR + NM - 3) / (NM - 2);   // conversion instructions per gap
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
                    __builtin_amdgcn_sched_group_barrier(0x200, PR, 0);                            // the LDS writes
                }
                __builtin_amdgcn_sched_barrier(0);
                rd(a0, b0, nxt, 0);
                mm(a1, b1);
                spread_half_step<PR * TB, PR + TB, 0>();
                wait_vmcnt_le<NB + 1>();                           // this wave's chunks of slab s + 2 and its tiles of slab s + 3 have landed
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

}  // namespace mlk
