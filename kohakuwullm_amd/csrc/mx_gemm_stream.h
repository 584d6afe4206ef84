// The persistent tile loop as ONE stream of K stages, fetched by waves of their own.
//
// A wave's vector memory operations retire in order, so a wave that both stores a tile and fetches the next one's operands waits for
// its stores before it may use what it fetched behind them.  persistent_gemm (mx_gemm_core.h) therefore works in rounds -- a K loop,
// then a burst of stores -- and with four to eight stages per tile the burst is as long as the K loop.  Here
//   * four loader waves issue every copy and nothing else, eight multiplying waves issue every store and nothing else: no wait for a
//     copy ever waits for a store, and the multiplying waves hold no copy offsets and issue no copies;
//   * operands go into a ring of four LDS slots, four stages ahead: the fragments of stage g + 1 are read into registers under the
//     MFMAs of stage g, so at the barrier that begins stage g its own slot is free again, and stage g + 4 goes there;
//   * results of 16 bits wait in registers, packed, and leave a quarter at a time under the first four steps of the next tile;
//   * the loaders have tiles of their own: while the last group of a tile is multiplied they fetch the next tile's first;
//   * scale bytes come as they lie in memory, 16 per row and group of four stages, and a lane reads the byte of its row's block from
//     there (ds_read_u8): no transposition and no shift.
// A tile is 128 x 128, eight waves as 4 (M) x 2 (N) of 32 x 64: three waves per SIMD leave 168 registers per lane, and 64 x 64 per wave
// spills at that.  0.43 us a stage with a tile on every CU (2.4 PFLOP/s), bound by the operand bytes between L2 and LDS; with the
// loads and stores in the same eight waves 98304 x 1024 x 512 in 64 experts took 109 us, without its stores 58; with loaders of their
// own 102 and 54, with the stores spread over the next tile's steps 72 (non-temporal; 107 if not).
// Operand layout, swizzle, the output run of a lane and the order in which a tile adds its K stages are those of mx_gemm_core.h: a tile
// that is not cut along K has the same bits.  Where the expert dW is cut, the ranges of stages follow from the tiles per expert, and the
// fp32 sums of the ranges are added in another order than 256 x 256 tiles have them in.
#pragma once

#include "mx_gemm_core.h"

namespace mx {

typedef GemmShape<128, 128, 4, 2> StreamShape;
constexpr int STREAM_LOADERS = 4;
constexpr int STREAM_THREADS = StreamShape::NTHR + 64 * STREAM_LOADERS;
constexpr int STREAM_SLOTS = 4;
constexpr int STREAM_SLOT_BYTES = StreamShape::DATA_A + StreamShape::DATA_B;
constexpr int STREAM_SCALES = STREAM_SLOTS * STREAM_SLOT_BYTES;               // where four buffers of scale bytes begin
constexpr int STREAM_SCALE_BYTES = 16 * (StreamShape::BM + StreamShape::BN);  // of a group of four stages
constexpr int STREAM_TILES = STREAM_SCALES + 4 * STREAM_SCALE_BYTES;          // where the tiles under way are described
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

// Both sides take a tile in an even number of steps, a step per stage and, behind an odd number of stages, an idle one, which
// fetches the last stage again and multiplies nothing: the fragments of a step are read into the one of two register sets that its
// parity names.  Step n uses slot n % 4.  Tiles have two steps at least, so the fetches of the next four steps reach into three
// groups of scale bytes at most, beside the one being multiplied: four buffers.

// The loader waves.  `P` provides Tile (four integers, the last one its stages), next(Tile &) and feed(Tile, loader, lane,
// StreamFeed &).
template <typename P>
__device__ __forceinline__ void stream_load(P &prob, uint8_t *smem, int loader) {
    typedef StreamShape S;
    constexpr int OPS = 8;
    const int lane = threadIdx.x & 63;
    typename P::Tile t;
    StreamFeed f;
    const uint32_t copy_to = __builtin_amdgcn_readfirstlane(lds_addr(smem) + loader * 4096);
    const uint32_t s_to = __builtin_amdgcn_readfirstlane(lds_addr(smem) + STREAM_SCALES + loader * 1024);
    int slot = 0, buf = 0, number = 0;  // bytes: the next step's slot, the next group's scale buffer; tiles so far
    int at = 0, steps = 0, total = 0;   // steps fetched and to fetch of the tile; of all tiles so far
    bool more = true;
    auto fetch = [&]() {  // the next step; with no tile left, what the last one fetched
        if (at == steps && more) {
            more = prob.next(t);
            if (loader == 0 && lane == 0) *(v4i *)(smem + STREAM_TILES + 16 * (number & 3)) = v4i{t.a, t.b, t.c, more ? t.stages : 0};
            number++;
            if (more) {
                prob.feed(t, loader, lane, f);
                at = 0, steps = (t.stages + 1) & ~1;
                total += steps;
            }
        }
        if (!total) return;  // a workgroup without tiles has nothing to fetch from
        if ((at & 3) == 0 && at < steps) {
            dma16(f.s, f.s_voff, s_to + buf);
            f.s += 16;
            buf = (buf + STREAM_SCALE_BYTES) & (4 * STREAM_SCALE_BYTES - 1);
        }
        dma16_run4(f.a, f.a_voff[0], f.a_voff[1], f.a_voff[2], f.a_voff[3], copy_to + slot);
        dma16_run4(f.b, f.b_voff[0], f.b_voff[1], f.b_voff[2], f.b_voff[3], copy_to + slot + S::DATA_A);
        slot = (slot + STREAM_SLOT_BYTES) & (STREAM_SLOTS * STREAM_SLOT_BYTES - 1);
        if (at < steps) at++;
        if (at < t.stages) f.a += f.a_ks, f.b += f.b_ks;
    };
#pragma unroll 1
    for (int s = 0; s < STREAM_SLOTS; s++) {
        fetch();
        if (!total) return;  // the multiplying waves have no tile either and have left
    }
    wait_vm_allow_c<(STREAM_SLOTS - 1) * OPS>();
    __syncthreads();
    // Four steps behind the fetches: at a step the next one has landed, and the one four on goes out into the slot of the one that
    // is being multiplied, whose fragments every wave has.
    for (int step = 0; more || step < total; step++) {
        wait_vm_allow_c<(STREAM_SLOTS - 2) * OPS>();
        __syncthreads();
        fetch();
    }
    wait_vm_allow_c<0>();  // copies that no step waited for must not land in the next workgroup's LDS
}

constexpr int STREAM_PARTS = 4;  // 16-byte parts of a lane's 16-bit results
template <int N>
using part = std::integral_constant<int, N>;

// The multiplying waves.  `P` provides WHOLE, whether every tile is in whole groups of four stages; if so pack(Lane, acc, parts) and
// store_part(Tile, Lane, n, part n), and if not store(Tile, Lane, acc).
template <typename P>
__device__ __forceinline__ void stream_multiply(P &prob, uint8_t *smem) {
    typedef StreamShape S;
    constexpr int SLOT_BYTES = STREAM_SLOT_BYTES;
    const Lane L = lane_of<S>();
    typename P::Tile t;
    if (!prob.next(t)) return;
    const int a_row = L.wm * S::WTM + L.r16, b_row = L.wn * S::WTN + L.r16;
    const int a_at = a_row * 128 + ((L.g ^ swz_a(a_row)) << 4), b_at = S::DATA_A + b_row * 128 + ((L.g ^ swz_a(b_row)) << 4);
    const uint8_t *const a_rd[2] = {smem + a_at, smem + (a_at ^ 64)}, *const b_rd[2] = {smem + b_at, smem + (b_at ^ 64)};
    // with constant slots, the upper two from bases of their own: an LDS read's offset is 16 bits
    int a_up_at[2] = {a_at + 2 * SLOT_BYTES, (a_at ^ 64) + 2 * SLOT_BYTES}, b_up_at[2] = {b_at + 2 * SLOT_BYTES, (b_at ^ 64) + 2 * SLOT_BYTES};
    asm volatile("" : "+v"(a_up_at[0]), "+v"(a_up_at[1]), "+v"(b_up_at[0]), "+v"(b_up_at[1]));
    const uint8_t *const a_up[2] = {smem + a_up_at[0], smem + a_up_at[1]}, *const b_up[2] = {smem + b_up_at[0], smem + b_up_at[1]};
    const uint8_t *const sa_rd = smem + STREAM_SCALES + a_row * 16 + L.g, *const sb_rd = smem + STREAM_SCALES + (S::BM + b_row) * 16 + L.g;
    // Fragments of a step and of the next one.  The first half of B's is held once: the next step's are read as soon as this step's
    // products of them are issued, and the registers that saves hold the tile that is being stored.
    static_assert(S::MT == 2 && S::NT == 4, "two products per fragment of B");
    struct Frags {
        v8i a[S::MT], b[S::NT / 2];
        int sa[S::MT], sb[S::NT];
    } fr[2];
    v8i b_once[S::NT / 2];
    auto read_fragment = [&](int slot, auto a_side, auto which, Frags &to) {
        constexpr bool A = a_side.value;
        constexpr int i = which.value;
        const bool up = P::WHOLE && slot >= 2 * SLOT_BYTES;
        const int off = i * 2048 + (up ? slot - 2 * SLOT_BYTES : slot);
        const v4i lo = *(const v4i *)((up ? A ? a_up[0] : b_up[0] : A ? a_rd[0] : b_rd[0]) + off);
        const v4i hi = *(const v4i *)((up ? A ? a_up[1] : b_up[1] : A ? a_rd[1] : b_rd[1]) + off);
        (A ? to.a[A ? i : 0] : i < S::NT / 2 ? b_once[A ? 0 : i & 1] : to.b[A ? 0 : i & 1]) = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    typedef std::true_type of_a;
    typedef std::false_type of_b;
    auto read_all = [&](int slot, Frags &to) {
        static_for<S::MT>([&](auto w) { read_fragment(slot, of_a{}, w, to); });
        static_for<S::NT>([&](auto w) { read_fragment(slot, of_b{}, w, to); });
    };
    auto read_scales = [&](int at, Frags &to) {
#pragma unroll
        for (int i = 0; i < S::MT; i++) to.sa[i] = (sa_rd + at)[i * 256];
#pragma unroll
        for (int j = 0; j < S::NT; j++) to.sb[j] = (sb_rd + at)[j * 256];
    };

    v4f acc[S::MT][S::NT];
    int half = 0, scales = 0, number = 0;  // bytes: the even step's slot, the current group's scale bytes; tiles so far
    auto next_group = [&]() { return (scales + STREAM_SCALE_BYTES) & (4 * STREAM_SCALE_BYTES - 1); };
    __syncthreads();
    read_all(0, fr[0]);
    read_scales(0, fr[0]);

    // A finished tile's results wait in registers, packed, and leave a part at a time under the first steps of the next one: the
    // CU's path to memory holds a few KB, and a burst of stores keeps the waves that issue it until memory has taken them.
    typename P::Tile held;
    v4i parts[STREAM_PARTS];
    int waiting = STREAM_PARTS;  // the first part that has not left; STREAM_PARTS: none
    auto release = [&](auto part) {
        if constexpr (P::WHOLE) {
            if (waiting != part.value) return;
            prob.store_part(held, L, part.value, parts[part.value]);
            waiting++;
        }
    };

    // One step, even or odd: its fragments are in fr[odd], the next step's are read into the other set.
    auto step = [&](auto odd, auto part, int next_slot, int next_scales, bool live) {
        Frags &now = fr[odd.value], &then = fr[odd.value ^ 1];
        __syncthreads();  // this step's fragments are in registers: its slot may be filled again; the next step has landed
        if constexpr (part.value < STREAM_PARTS) release(part);
        if (live) {
            static_for<S::MT * S::NT>([&](auto at) {
                constexpr int i = at.value % S::MT, j = at.value / S::MT;
                const v8i &bj = j < S::NT / 2 ? b_once[j & 1] : now.b[j & 1];
                acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(now.a[i], bj, acc[i][j], 0, 0, 0, now.sa[i], 0, now.sb[j]);
                if constexpr (at.value < 2) read_fragment(next_slot, of_a{}, at, then);
                if constexpr (at.value == 1 || at.value == 3) read_fragment(next_slot, of_b{}, std::integral_constant<int, at.value / 2>{}, then);
                if constexpr (at.value == 2) read_fragment(next_slot, of_b{}, std::integral_constant<int, 2>{}, then);
                if constexpr (at.value == 4) read_fragment(next_slot, of_b{}, std::integral_constant<int, 3>{}, then);
                if constexpr (at.value == 5) read_scales(next_scales, then);
                __builtin_amdgcn_sched_barrier(0);
            });
        } else {
            read_all(next_slot, then);
            read_scales(next_scales, then);
        }
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
        typedef std::integral_constant<int, 0> even;
        typedef std::integral_constant<int, 1> odd;
        typedef part<STREAM_PARTS> none;
        if constexpr (P::WHOLE) {  // whole groups begin with slot 0: slots are constants
            for (int k = 0; k < stages; k += 4) {
                step(even{}, part<0>{}, SLOT_BYTES, scales + 4, true);
                step(odd{}, part<1>{}, 2 * SLOT_BYTES, scales + 8, true);
                step(even{}, part<2>{}, 3 * SLOT_BYTES, scales + 12, true);
                scales = next_group();
                step(odd{}, part<3>{}, 0, scales, true);
            }
        } else {
            for (int k = 0; k < stages; k += 2) {
                step(even{}, none{}, half + SLOT_BYTES, scales + 4 * (k & 3) + 4, true);
                // behind the odd step comes the group's second half, the next group's first stage, or the next tile's
                const bool ends = (k & 2) || k + 2 >= stages;
                const int from = ends ? next_group() : scales;
                half ^= 2 * SLOT_BYTES;
                step(odd{}, none{}, half, ends ? from : scales + 8, k + 1 < stages);
                scales = from;
            }
        }
        if constexpr (P::WHOLE) {  // K of four stages and more: every part of the tile before has left
            held = t, waiting = 0;
            prob.pack(L, acc, parts);
        } else {
            prob.store(t, L, acc);
        }
        // the next tile, as the loaders described it when they began to fetch it
        number++;
        const v4i d = *(const v4i *)(smem + STREAM_TILES + 16 * (number & 3));
        t.a = __builtin_amdgcn_readfirstlane(d[0]), t.b = __builtin_amdgcn_readfirstlane(d[1]), t.c = __builtin_amdgcn_readfirstlane(d[2]);
        stages = t.stages = __builtin_amdgcn_readfirstlane(d[3]);
    } while (stages);
    if constexpr (P::WHOLE) static_for<STREAM_PARTS>([&](auto n) { release(n); });
}

// A lane's 16-bit results in parts of 16 bytes.  Neighbouring lanes swap half of every two rows, so that a part is 16 bytes of one row
// instead of 8 of two: a store costs the CU's one path to memory 12 clocks whatever it carries (32 KB in stores of 8 bytes a lane 760
// clocks, of 16 bytes 415).
template <int CDT>
__device__ __forceinline__ void stream_pack(const Lane &L0, v4f (&acc)[StreamShape::MT][StreamShape::NT], v4i (&parts)[STREAM_PARTS]) {
    typedef StreamShape S;
    static_assert(S::NT == 4 && S::MT * 2 == STREAM_PARTS, "four consecutive columns per lane");
    const Lane L = opaque(L0);
    const bool odd = L.lane & 1;
    auto pack = [](float lo, float hi) -> uint32_t {
        if (CDT == MX_BF16) return pack2_bf16(lo, hi);
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        const h2 h = {(_Float16)lo, (_Float16)hi};
        return __builtin_bit_cast(uint32_t, h);
    };
#pragma unroll
    for (int i = 0; i < S::MT; i++)
#pragma unroll
        for (int v = 0; v < 4; v += 2) {
            v4i w;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int first = (int)pack(acc[i][2 * h][v], acc[i][2 * h + 1][v]), second = (int)pack(acc[i][2 * h][v + 1], acc[i][2 * h + 1][v + 1]);
                const int other = __builtin_amdgcn_mov_dpp(odd ? first : second, 0xB1, 0xF, 0xF, true);  // lane ^ 1
                w[h] = odd ? other : first;
                w[2 + h] = odd ? second : other;
            }
            parts[2 * i + v / 2] = w;
        }
}

// Stores part n of them, where it lies inside rows [row0, row_end) and columns [col0, col_end) (col_end % 8 == 0; rows on 16 bytes).
// HINT: non-temporal, for results that nothing reads soon (dW of 1024 x 512, 33000 rows in 64 experts, 49.6 -> 38.6 us).
template <bool HINT>
__device__ __forceinline__ void stream_store_part(void *out, int64_t ld, int row0, int row_end, int col0, int col_end, const Lane &L0, int n,
                                                  const v4i &part) {
    typedef StreamShape S;
    const Lane L = opaque(L0);
    const int row = row0 + L.wm * S::WTM + 4 * (L.lane >> 4) + (L.lane & 1) + 16 * (n >> 1) + 2 * (n & 1), col = col0 + L.wn * S::WTN + 8 * ((L.lane & 15) >> 1);
    if (row < row_end && col < col_end) stream_store<HINT>((v4i *)((uint16_t *)out + (int64_t)row * ld + col), part);
}

// Stores a tile's rows [row0, row_end) and columns [col0, col_end) of a matrix: 16-byte runs (col_end % 8 == 0, fp32: % 4; rows on
// 16 bytes).
template <int CDT>
__device__ __forceinline__ void stream_store_tile(void *out, int64_t ld, int row0, int row_end, int col0, int col_end, const Lane &L0,
                                                  v4f (&acc)[StreamShape::MT][StreamShape::NT]) {
    typedef StreamShape S;
    static_assert(S::NT == 4, "four consecutive columns per lane");
    const Lane L = opaque(L0);
    if constexpr (CDT == MX_FP32) {
        const int row = row0 + L.wm * S::WTM + 4 * (L.lane >> 4), col = col0 + L.wn * S::WTN + 4 * (L.lane & 15);
        const int rows = col < col_end ? row_end - row : 0;
        float *const at = (float *)out + (int64_t)row * ld + col;
#pragma unroll
        for (int i = 0; i < S::MT; i++)
#pragma unroll
            for (int v = 0; v < 4; v++)
                if (16 * i + v < rows)
                    stream_store<true>((v4f *)(at + (int64_t)(16 * i + v) * ld), v4f{acc[i][0][v], acc[i][1][v], acc[i][2][v], acc[i][3][v]});
    } else {
        v4i parts[STREAM_PARTS];
        stream_pack<CDT>(L, acc, parts);
#pragma unroll
        for (int n = 0; n < STREAM_PARTS; n++) stream_store_part<true>(out, ld, row0, row_end, col0, col_end, L, n, parts[n]);
    }
}

}  // namespace mx
