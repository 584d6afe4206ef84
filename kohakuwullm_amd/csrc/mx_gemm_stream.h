// The persistent tile loop as ONE stream of K stages, fetched by waves of their own.
//
// A wave's vector memory operations retire in order, so a wave that both stores a tile and fetches the next one's operands waits for
// its stores before it may use what it fetched behind them.  persistent_gemm (mx_gemm_core.h) therefore works in rounds -- a K loop,
// then a burst of stores -- and with four to eight stages per tile the burst is as long as the K loop.  Here
//   * four loader waves issue every copy and nothing else, eight multiplying waves issue every store and nothing else: no wait for a
//     copy ever waits for a store, and the multiplying waves hold no copy offsets and issue no copies;
//   * operands go into a ring of four LDS slots, four stages ahead: the fragments of stage g + 1 are read into registers under the
//     MFMAs of stage g, so at the barrier that begins stage g its own slot is free again, and stage g + 4 goes there;
//   * the loaders have tiles of their own: while the last group of a tile is multiplied they fetch the next tile's first;
//   * scale bytes come as they lie in memory, 16 per row and group of four stages, and a lane reads the byte of its row's block from
//     there (ds_read_u8): no transposition and no shift.
// A tile is 128 x 128, eight waves as 4 (M) x 2 (N) of 32 x 64: three waves per SIMD leave 168 registers per lane, and 64 x 64 per wave
// spills at that.  0.43 us a stage with a tile on every CU (2.4 PFLOP/s), bound by the operand bytes between L2 and LDS; with the
// loads and stores in the same eight waves 98304 x 1024 x 512 in 64 experts took 109 us, without its stores 58; here 102 and 54.
// Operand layout, swizzle, the output run of a lane and the order of the sums are those of mx_gemm_core.h: the same bits.
#pragma once

#include "mx_gemm_core.h"

namespace mx {

typedef GemmShape<128, 128, 4, 2> StreamShape;
constexpr int STREAM_LOADERS = 4;
constexpr int STREAM_THREADS = StreamShape::NTHR + 64 * STREAM_LOADERS;
constexpr int STREAM_SLOTS = 4;
constexpr int STREAM_SLOT_BYTES = StreamShape::DATA_A + StreamShape::DATA_B;
constexpr int STREAM_SCALE_BYTES = 16 * (StreamShape::BM + StreamShape::BN);  // of a group of four stages
constexpr int STREAM_TILES = STREAM_SLOTS * STREAM_SLOT_BYTES + 2 * STREAM_SCALE_BYTES;  // where the tiles under way are described
constexpr int STREAM_LDS_BYTES = STREAM_TILES + 4 * 16;

// What a loader wave's next copies read: wave-uniform bases (biased, see dma16_run2) and the lane's offsets from them, for the four
// 8-row chunks of A and of B that are the wave's, and for the lane's row of scale bytes.
struct StreamFeed {
    const uint8_t *a, *b, *s;
    int64_t a_ks, b_ks;  // bytes from one stage of an operand to the next
    uint32_t a_voff[4], b_voff[4], s_voff;
};

// LDS row, in the tile image of A or of B, of this lane's 16-byte chunk of a loader's copy q.
__device__ __forceinline__ int stream_row(int loader, int lane, int q) { return (loader * 4 + q) * 8 + (lane >> 3); }

// The loader waves.  `P` provides Tile (four integers, the last one its stages, whole groups of four), next(Tile &) and
// feed(Tile, loader, lane, StreamFeed &).
template <typename P>
__device__ __forceinline__ void stream_load(P &prob, uint8_t *smem, int loader) {
    typedef StreamShape S;
    constexpr int OPS = 8;
    const int lane = threadIdx.x & 63;
    typename P::Tile t;
    StreamFeed f;
    const uint32_t copy_to = __builtin_amdgcn_readfirstlane(lds_addr(smem) + loader * 4096);
    const uint32_t s_to = __builtin_amdgcn_readfirstlane(lds_addr(smem) + STREAM_SLOTS * STREAM_SLOT_BYTES + loader * 1024);
    int buf = 0, number = 0, left = 0;  // scale buffer, tiles so far, stages of the tile still to fetch
    auto advance = [&]() -> bool {
        if (left) return true;
        const bool more = prob.next(t);
        if (loader == 0 && lane == 0) *(v4i *)(smem + STREAM_TILES + 16 * (number & 3)) = v4i{t.a, t.b, t.c, more ? t.stages : 0};
        number++;
        if (!more) return false;
        prob.feed(t, loader, lane, f);
        left = t.stages;
        return true;
    };
    auto fetch = [&](auto sc) {  // stage sc of a group
        constexpr int s = sc.value;
        if constexpr (s == 0) {
            dma16(f.s, f.s_voff, s_to + buf);
            f.s += 16;
            buf ^= STREAM_SCALE_BYTES;
            left -= 4;
        }
        dma16_run4(f.a, f.a_voff[0], f.a_voff[1], f.a_voff[2], f.a_voff[3], copy_to + s * STREAM_SLOT_BYTES);
        dma16_run4(f.b, f.b_voff[0], f.b_voff[1], f.b_voff[2], f.b_voff[3], copy_to + s * STREAM_SLOT_BYTES + S::DATA_A);
        f.a += f.a_ks, f.b += f.b_ks;
    };
    if (!advance()) return;
    static_for<4>([&](auto s) { fetch(s); });
    wait_vm_allow_c<3 * OPS>();
    __syncthreads();
    // Group after group, one behind the fetches: at stage s the next stage has landed, and stage s of the next group goes out into
    // the slot of the stage that is being multiplied, whose fragments every wave has.
    while (advance()) {
        static_for<4>([&](auto s) {
            wait_vm_allow_c<2 * OPS>();
            __syncthreads();
            fetch(s);
        });
    }
    static_for<4>([&](auto s) {
        wait_vm_allow_c<(s.value < 2 ? 2 - s.value : 0) * OPS>();
        __syncthreads();
    });
}

// The multiplying waves.  `P` provides store(Tile, Lane, acc).
template <typename P>
__device__ __forceinline__ void stream_multiply(P &prob, uint8_t *smem) {
    typedef StreamShape S;
    constexpr int SLOT_BYTES = STREAM_SLOT_BYTES, SCALES = STREAM_SLOTS * STREAM_SLOT_BYTES;
    const Lane L = lane_of<S>();
    typename P::Tile t;
    if (!prob.next(t)) return;
    // LDS read bases: slots 0 and 1 within the 16-bit offset of an LDS read, slots 2 and 3 from a second set 64 KB on
    const int a_row = L.wm * S::WTM + L.r16, b_row = L.wn * S::WTN + L.r16;
    const int a_at = a_row * 128 + ((L.g ^ swz_a(a_row)) << 4), b_at = S::DATA_A + b_row * 128 + ((L.g ^ swz_a(b_row)) << 4);
    const uint8_t *a_rd[2][2], *b_rd[2][2];
#pragma unroll
    for (int half = 0; half < 2; half++) {
        const uint8_t *const base = smem + half * 2 * SLOT_BYTES;
        a_rd[half][0] = base + a_at, a_rd[half][1] = base + (a_at ^ 64);
        b_rd[half][0] = base + b_at, b_rd[half][1] = base + (b_at ^ 64);
    }
    const uint8_t *const sa_rd = smem + SCALES + a_row * 16 + L.g, *const sb_rd = smem + SCALES + (S::BM + b_row) * 16 + L.g;
    struct Frags {
        v8i a[S::MT], b[S::NT];
        int sa[S::MT], sb[S::NT];
    } fr[2];
    auto read_fragment = [&](auto slot, auto which, Frags &to) {  // A rows first, then B rows
        constexpr int off = (slot.value & 1) * SLOT_BYTES, half = slot.value >> 1;
        constexpr bool A = which.value < S::MT;
        constexpr int i = A ? which.value : which.value - S::MT;
        const uint8_t *const(&at)[2] = A ? a_rd[half] : b_rd[half];
        const v4i lo = *(const v4i *)(at[0] + off + i * 2048), hi = *(const v4i *)(at[1] + off + i * 2048);
        (A ? to.a[A ? i : 0] : to.b[A ? 0 : i]) = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    auto read_scales = [&](int at, Frags &to) {
#pragma unroll
        for (int i = 0; i < S::MT; i++) to.sa[i] = (sa_rd + at)[i * 256];
#pragma unroll
        for (int j = 0; j < S::NT; j++) to.sb[j] = (sb_rd + at)[j * 256];
    };

    v4f acc[S::MT][S::NT];
    int buf = 0, number = 0;  // where the scale bytes of the current group lie, tiles so far
    __syncthreads();
    static_for<S::MT + S::NT>([&](auto w) { read_fragment(std::integral_constant<int, 0>{}, w, fr[0]); });
    read_scales(0, fr[0]);

    // Stage s of a group: its fragments are in fr[s & 1], the next stage's are read into the other set.
    auto stage = [&](auto sc) {
        constexpr int s = sc.value;
        typedef std::integral_constant<int, (s + 1) & 3> after;
        Frags &now = fr[s & 1], &then = fr[(s + 1) & 1];
        const int scales = (s == 3 ? buf ^ STREAM_SCALE_BYTES : buf) + 4 * after::value;
        __syncthreads();  // this stage's fragments are in registers: its slot may be filled again, and the next stage has landed
        static_for<S::MT * S::NT>([&](auto step) {
            constexpr int i = step.value % S::MT, j = step.value / S::MT;
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(now.a[i], now.b[j], acc[i][j], 0, 0, 0, now.sa[i], 0, now.sb[j]);
            if constexpr (step.value < S::MT + S::NT) read_fragment(after{}, step, then);
            if constexpr (step.value == S::MT + S::NT) read_scales(scales, then);
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (s == 3) buf ^= STREAM_SCALE_BYTES;
#pragma unroll
        for (int i = 0; i < S::MT; i++)
#pragma unroll
            for (int j = 0; j < S::NT; j++) asm volatile("" : "+v"(acc[i][j]));  // in front of the next barrier, not behind it
    };
    int stages = t.stages;
    do {
#pragma unroll
        for (int i = 0; i < S::MT; i++)
#pragma unroll
            for (int j = 0; j < S::NT; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
        for (int left = stages; left; left -= 4) static_for<4>([&](auto s) { stage(s); });
        prob.store(t, L, acc);
        // the next tile, as the loaders described it when they began to fetch it
        number++;
        const v4i d = *(const v4i *)(smem + STREAM_TILES + 16 * (number & 3));
        t.a = __builtin_amdgcn_readfirstlane(d[0]), t.b = __builtin_amdgcn_readfirstlane(d[1]), t.c = __builtin_amdgcn_readfirstlane(d[2]);
        stages = t.stages = __builtin_amdgcn_readfirstlane(d[3]);
    } while (stages);
}

}  // namespace mx
