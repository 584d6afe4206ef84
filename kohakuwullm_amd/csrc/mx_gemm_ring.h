// The MXFP8 NT GEMM on 128 x 128 tiles behind a four-slot ring of K stages, for products whose 256 x 256 tiles (mx_gemm_core.h)
// leave most of the chip idle.
//
// Such a launch is not bound by a rate but by one workgroup's walk along K: with fewer tiles than CUs every CU owns one
// tile, and what counts is how long a stage takes when nothing else hides its latencies.  The persistent kernel fetches one
// stage ahead and reads its fragments after the stage's barrier (1.35 us per stage of 256 x 256 x 128 on a lone CU, 0.6 of
// it MFMA).  Here
//   * a tile is a quarter of that, so a product has four times as many workgroups, and K may be cut into slices on top
//     (fp32 partial tiles, added by slice_reduce);
//   * operands are fetched three stages ahead into a ring of four 32 KB slots (128 of the CU's 160 KB), so a copy has three
//     stage times to land and the stage-ending wait is for one issued long ago;
//   * the fragments of the next stage are read from LDS into a second register set between the MFMAs of the current one: the
//     MFMA pipe waits for the barrier, not for LDS;
//   * scale bytes travel through the copy engine as they lie in memory, 16 bytes per row and four stages, and a lane shifts
//     its row's word to its block's byte, six shifts per stage, instead of a transposition;
//   * the four stages of a group are unrolled, with slots, wait counts and scale offsets as constants: a wave issues at most
//     one instruction per four clocks, and the address arithmetic of a stage written for any slot (135 instructions per wave
//     and stage) cost as much as its MFMAs.
// Eight waves as 4 (M) x 2 (N), 32 x 64 each, two per SIMD.  Operand layout, swizzle, output run per lane and the MFMA are those of
// mx_gemm_core.h; the results are the same bits wherever K is not cut.  K is in whole stages of 128.  A tile or K
// slice that ends inside a group of four keeps the schedule of a whole one -- a copy past its last stage fetches that stage
// again, so that the wait counts hold -- and leaves the absent stages' MFMAs out; the 16 scale bytes per row of such a group
// are the last 16 of the row instead of the next 16, which would run past the matrix, and its stages read that much further on.  Products of one to three stages, whose rows have no 16 scale bytes, have a
// walk of their own (ring_gemm_short): there is nothing to pipeline in them.
#pragma once

#include "mx_gemm_core.h"

namespace mx {

typedef GemmShape<128, 128, 4, 2> RingShape;
constexpr int RING_SLOTS = 4;
constexpr int RING_SLOT_BYTES = RingShape::DATA_A + RingShape::DATA_B;
constexpr int RING_SCALE_BYTES = 16 * (RingShape::BM + RingShape::BN);  // of a group of four stages
constexpr int RING_LDS_BYTES = RING_SLOTS * RING_SLOT_BYTES + 2 * RING_SCALE_BYTES;

// Two copies behind one write of M0 = `lds` + OFF (see dma16_run2).
template <int OFF>
__device__ __forceinline__ void ring_copy2(const uint8_t *biased_base, uint32_t v0, uint32_t v1, uint32_t lds) {
    asm volatile("s_add_u32 m0, %3, %4\n\ts_nop 0\n\t"
                 "global_load_lds_dwordx4 %0, %2\n\t"
                 "global_load_lds_dwordx4 %1, %2 offset:1024"
                 :
                 : "v"(v0), "v"(v1), "s"(biased_base), "s"(lds), "n"(OFF)
                 : "memory", "scc");
}

// One copy of 4 bytes per lane to LDS address `lds`, 256 bytes in a row.
__device__ __forceinline__ void dma4(const uint8_t *base, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" : : "v"(voff), "s"(base), "s"(lds) : "memory");
}

template <typename P>
__device__ __forceinline__ void ring_gemm(P &prob, uint8_t *smem) {
    typedef RingShape S;
    static_assert(S::QA == 2 && S::QB == 2 && RING_SLOTS == 4, "one run of two copies per operand, wave and stage");
    constexpr int OPS = 4;  // vector-memory operations every wave issues per stage (scale copies come on top, in some waves)
    const Lane L = lane_of<S>();
    typename P::Tile t;
    if (!prob.next(t)) return;
    IssueCtx<S> c;
    prob.context(t, L, c);
    const int stages = c.kt1 - c.kt0, groups = (stages + 3) >> 2, last = stages - 4 * (groups - 1);  // stages of the last group
    const int shift = 4 * (4 - last);  // bytes its scale words begin in front of its first stage

    // LDS read bases: slots 0 and 1 within the 16-bit offset of an LDS read, slots 2 and 3 from a second set 64 KB on
    const int a_row = L.wm * S::WTM + L.r16, b_row = L.wn * S::WTN + L.r16;
    const uint8_t *a_rd[2][2], *b_rd[2][2];
#pragma unroll
    for (int half = 0; half < 2; half++) {
        const uint8_t *const base = smem + half * 2 * RING_SLOT_BYTES;
        a_rd[half][0] = base + a_row * 128 + ((L.g ^ swz_a(a_row)) << 4);
        a_rd[half][1] = base + (a_row * 128 + (((L.g ^ swz_a(a_row)) << 4) ^ 64));
        b_rd[half][0] = base + S::DATA_A + b_row * 128 + ((L.g ^ swz_a(b_row)) << 4);
        b_rd[half][1] = base + S::DATA_A + (b_row * 128 + (((L.g ^ swz_a(b_row)) << 4) ^ 64));
    }
    const uint8_t *const sa_rd = smem + RING_SLOTS * RING_SLOT_BYTES + a_row * 16;
    const uint8_t *const sb_rd = smem + RING_SLOTS * RING_SLOT_BYTES + (S::BM + b_row) * 16;
    int scale_at = 0;  // which of the two scale buffers the current group reads

    // what the next copies fetch: the A and B rows of a stage, the scale words of a group
    const uint8_t *ga = uniform_ptr(c.a_base + (int64_t)c.kt0 * c.a_ks - COPY_BIAS);
    const uint8_t *gb = uniform_ptr(c.b_base + (int64_t)c.kt0 * c.b_ks - COPY_BIAS);
    const bool scale_wave = L.wave < (S::BM + S::BN) / 64;
    const uint8_t *gs = uniform_ptr((L.wave < S::BM / 64 ? c.sa_base : c.sb_base) + 4 * c.kt0 - (groups == 1 ? shift : 0));
    int left = stages;  // to fetch
    const uint32_t copy_to = __builtin_amdgcn_readfirstlane(lds_addr(smem) + L.wave * S::QA * 1024);
    const uint32_t scales_to = __builtin_amdgcn_readfirstlane(lds_addr(smem) + RING_SLOTS * RING_SLOT_BYTES + L.wave * 1024);
    auto copy_a = [&](auto slot) {
        ring_copy2<slot.value * RING_SLOT_BYTES>(ga, c.a_voff[0], c.a_voff[1], copy_to);
        ga += left > 1 ? c.a_ks : 0;
    };
    auto copy_b = [&](auto slot) {
        ring_copy2<slot.value * RING_SLOT_BYTES + S::DATA_A>(gb, c.b_voff[0], c.b_voff[1], copy_to);
        gb += left > 1 ? c.b_ks : 0;
        left--;
    };
    auto copy_scales = [&](int buffer) {
        if (scale_wave) dma16(gs, c.s_voff, scales_to + buffer * RING_SCALE_BYTES);
    };

    struct Frags {
        v8i a[S::MT], b[S::NT];
        int sa[S::MT], sb[S::NT];
    };
    auto read_fragment = [&](auto slot, auto which, Frags &f) {  // A rows first, then B rows
        constexpr int off = (slot.value & 1) * RING_SLOT_BYTES, half = slot.value >> 1;
        if constexpr (which.value < S::MT) {
            const v4i lo = *(const v4i *)(a_rd[half][0] + off + which.value * 2048), hi = *(const v4i *)(a_rd[half][1] + off + which.value * 2048);
            f.a[which.value] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        } else {
            constexpr int j = which.value - S::MT;
            const v4i lo = *(const v4i *)(b_rd[half][0] + off + j * 2048), hi = *(const v4i *)(b_rd[half][1] + off + j * 2048);
            f.b[j] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        }
    };
    auto read_scales = [&](auto slot, int at, Frags &f) {  // `at`: where the group's first stage lies in the scale buffers
        const int off = at + 4 * slot.value;
#pragma unroll
        for (int i = 0; i < S::MT; i++) f.sa[i] = *(const int *)(sa_rd + off + i * 256);
#pragma unroll
        for (int j = 0; j < S::NT; j++) f.sb[j] = *(const int *)(sb_rd + off + j * 256);
    };

    v4f acc[S::MT][S::NT];
#pragma unroll
    for (int i = 0; i < S::MT; i++)
#pragma unroll
        for (int j = 0; j < S::NT; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

    copy_scales(0);
    static_for<3>([&](auto s) {
        copy_a(s);
        copy_b(s);
    });
    wait_vm_allow_c<2 * OPS>();
    __syncthreads();
    Frags f[2];
    static_for<S::MT + S::NT>([&](auto w) { read_fragment(std::integral_constant<int, 0>{}, w, f[0]); });
    read_scales(std::integral_constant<int, 0>{}, groups == 1 ? shift : 0, f[0]);

    // Stage s of a group (slot s).  Stage s + 1 has landed everywhere behind the wait and the barrier; stage s + 3 goes out
    // into the slot stage s - 1 was read from (every wave had those fragments in registers before this barrier); the
    // fragments of s + 1 are read into `then`; the MFMAs run on `now`, read a stage ago.  `then_at`: where the scale words of the
    // next group lie.  TAIL: the tile's last group, where only its own last stage is left to fetch.
    auto stage = [&](auto sc, auto tail, Frags &now, Frags &then, int now_at, int then_at) {
        constexpr int s = sc.value;
        constexpr bool TAIL = tail.value, NEXT = !TAIL || s < 3, FETCH = !TAIL || s == 0;
        typedef std::integral_constant<int, (s + 1) & 3> next_slot;
        typedef std::integral_constant<int, (s + 3) & 3> free_slot;
        if constexpr (NEXT) {
            wait_vm_allow_c<TAIL && s == 2 ? 0 : OPS>();
            __syncthreads();
        }
        // the byte of the lane's block (shifted here, not where the word is read: that would wait for the word)
        int sa[S::MT], sb[S::NT];
#pragma unroll
        for (int i = 0; i < S::MT; i++) sa[i] = (int)((uint32_t)now.sa[i] >> (8 * L.g));
#pragma unroll
        for (int j = 0; j < S::NT; j++) sb[j] = (int)((uint32_t)now.sb[j] >> (8 * L.g));
        static_for<S::MT * S::NT>([&](auto step) {
            constexpr int i = step.value % S::MT, j = step.value / S::MT;
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(now.a[i], now.b[j], acc[i][j], 0, 0, 0, sa[i], 0, sb[j]);
            if constexpr (NEXT && step.value < S::MT + S::NT) read_fragment(next_slot{}, step, then);
            if constexpr (NEXT && step.value == S::MT + S::NT) read_scales(next_slot{}, s == 3 ? then_at : now_at, then);
            if constexpr (FETCH && step.value == 1) {
                if constexpr (s == 1) copy_scales(scale_at ^ 1);  // with the first stage of the next group
                copy_a(free_slot{});
            }
            if constexpr (FETCH && step.value == 5) copy_b(free_slot{});
            __builtin_amdgcn_sched_barrier(0);
        });
#pragma unroll
        for (int i = 0; i < S::MT; i++)
#pragma unroll
            for (int j = 0; j < S::NT; j++) asm volatile("" : "+v"(acc[i][j]));  // in front of the next barrier, not behind it
    };
    for (int g = 1; g < groups; g++) {
        const int back = g + 1 == groups ? shift : 0;  // the next group is the last one
        const int now_at = scale_at * RING_SCALE_BYTES, then_at = (scale_at ^ 1) * RING_SCALE_BYTES + back;
        gs += 16 - back;
        stage(std::integral_constant<int, 0>{}, std::false_type{}, f[0], f[1], now_at, then_at);
        stage(std::integral_constant<int, 1>{}, std::false_type{}, f[1], f[0], now_at, then_at);
        stage(std::integral_constant<int, 2>{}, std::false_type{}, f[0], f[1], now_at, then_at);
        stage(std::integral_constant<int, 3>{}, std::false_type{}, f[1], f[0], now_at, then_at);
        scale_at ^= 1;
    }
    const int tail_at = scale_at * RING_SCALE_BYTES + shift;
    stage(std::integral_constant<int, 0>{}, std::true_type{}, f[0], f[1], tail_at, 0);
    if (last > 1) stage(std::integral_constant<int, 1>{}, std::true_type{}, f[1], f[0], tail_at, 0);
    if (last > 2) stage(std::integral_constant<int, 2>{}, std::true_type{}, f[0], f[1], tail_at, 0);
    if (last > 3) stage(std::integral_constant<int, 3>{}, std::true_type{}, f[1], f[0], tail_at, 0);
    wait_vm_allow_c<0>();  // copies that no stage waited for must not land in the next workgroup's LDS
    prob.epilogue(t, L, acc, LdsScratch{smem, smem, smem});
}

// K of one to three stages (the token axis of a short batch): all of them are fetched, waited for once and multiplied.  Scale
// words come one dword per row and stage, [stage][row].  us on the 256 x 256 tiles, whose scale bytes go through registers
// there, and here: fp32 dW of 2048 x 2048 over 128 / 384 tokens 13.2 / 16.0 and 7.8 / 8.9; both gradients of a 512 -> 1536 layer
// over 128 tokens 15.6 and 8.2.
template <typename P>
__device__ __forceinline__ void ring_gemm_short(P &prob, uint8_t *smem) {
    typedef RingShape S;
    const Lane L = lane_of<S>();
    typename P::Tile t;
    if (!prob.next(t)) return;
    IssueCtx<S> c;
    prob.context(t, L, c);
    const int stages = c.kt1 - c.kt0;
    const uint32_t copy_to = __builtin_amdgcn_readfirstlane(lds_addr(smem) + L.wave * S::QA * 1024);
    const uint32_t scales_to = __builtin_amdgcn_readfirstlane(lds_addr(smem) + RING_SLOTS * RING_SLOT_BYTES + L.wave * 256);
    static_for<3>([&](auto s) {
        if (s.value >= stages) return;
        const int kt = c.kt0 + s.value;
        ring_copy2<s.value * RING_SLOT_BYTES>(uniform_ptr(c.a_base + kt * c.a_ks - COPY_BIAS), c.a_voff[0], c.a_voff[1], copy_to);
        ring_copy2<s.value * RING_SLOT_BYTES + S::DATA_A>(uniform_ptr(c.b_base + kt * c.b_ks - COPY_BIAS), c.b_voff[0], c.b_voff[1], copy_to);
        if (L.wave < (S::BM + S::BN) / 64)
            dma4(uniform_ptr((L.wave < S::BM / 64 ? c.sa_base : c.sb_base) + 4 * kt), c.s_voff, scales_to + s.value * 4 * (S::BM + S::BN));
    });
    v4f acc[S::MT][S::NT];
#pragma unroll
    for (int i = 0; i < S::MT; i++)
#pragma unroll
        for (int j = 0; j < S::NT; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    const int a_row = L.wm * S::WTM + L.r16, b_row = L.wn * S::WTN + L.r16;
    wait_vm_allow_c<0>();
    __syncthreads();
    for (int s = 0; s < stages; s++) {
        const uint8_t *const la = smem + s * RING_SLOT_BYTES, *const lb = la + S::DATA_A;
        const uint32_t *const scales = (const uint32_t *)(smem + RING_SLOTS * RING_SLOT_BYTES) + s * (S::BM + S::BN);
        auto fragment = [&](const uint8_t *tile, int row) {
            const uint8_t *const at = tile + row * 128;
            const int chunk = (L.g ^ swz_a(row)) << 4;
            const v4i lo = *(const v4i *)(at + chunk), hi = *(const v4i *)(at + (chunk ^ 64));
            return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        };
        v8i a[S::MT];
        int sa[S::MT];
#pragma unroll
        for (int i = 0; i < S::MT; i++) a[i] = fragment(la, a_row + 16 * i), sa[i] = (int)(scales[a_row + 16 * i] >> (8 * L.g));
#pragma unroll
        for (int j = 0; j < S::NT; j++) {
            const v8i b = fragment(lb, b_row + 16 * j);
            const int sb = (int)(scales[S::BM + b_row + 16 * j] >> (8 * L.g));
#pragma unroll
            for (int i = 0; i < S::MT; i++)
                acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a[i], b, acc[i][j], 0, 0, 0, sa[i], 0, sb);
        }
    }
    prob.epilogue(t, L, acc, LdsScratch{smem, smem, smem});
}

}  // namespace mx
