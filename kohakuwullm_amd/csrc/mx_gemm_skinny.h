// The MXFP8 NT GEMM for a few rows of A (sequences being decoded): the weights are read once and little else costs.
//
// Tiles of 128 columns leave most of the chip without a share of the weights (2048 -> 3072: 24 workgroups), and each walks all
// of K alone.  Here a workgroup owns 16 columns -- one 16-column sub-tile of the MFMA -- and its eight waves take an eighth of
// the K stages each.  A wave fetches U of its stages at once into LDS of its own and waits for its own copies only: one memory round
// trip per 1024 U of K.  The eight partial sums meet in LDS, behind two barriers, and are added in wave order.
// The copy engine brings the operands although no wave shares them: it fetches a row's 128 bytes with eight neighbouring lanes,
// where loads straight into the MFMA's operand registers have 16 bytes of another row in every neighbouring lane, which the
// texture path takes at about 12 B per clock (64 rows of A: 10 us of a 10 us launch).
#pragma once

#include "mx_gemm_core.h"

namespace mx {

constexpr int SKINNY_WAVES = 8, SKINNY_N = 16;
constexpr int SRC_CODES = -1;  // A is quantized; else the type of the activations that are quantized on the way
__host__ __device__ constexpr int skinny_stage_bytes(int mt) { return (mt + 1) * 16 * 128; }
// ... and, for activations, the scale words of the stage's rows
__host__ __device__ constexpr int skinny_lds_bytes(int src, int mt, int u) {
    return SKINNY_WAVES * u * (skinny_stage_bytes(mt) + (src == SRC_CODES ? 0 : 16 * mt * 4));
}

// MT: sub-tiles of 16 rows; U: K stages a wave has in flight.  SRC: where A comes from.  With activations (`p.aq` are they, `p.lda`
// their pitch in elements) the row quantizer's launch and its round trip through memory go away: every workgroup quantizes the
// rows again, a K stage of four rows per load, as mx_quantize_rows does -- the same bytes.
template <int CDT, int MT, int U, int SRC, int CAST, typename Args>
__device__ __forceinline__ void skinny_gemm(const Args &p, int tile, uint8_t *smem) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, g = lane >> 4, n0 = tile * SKINNY_N;
    const int KT = p.K >> 7, per = (KT + SKINNY_WAVES - 1) / SKINNY_WAVES;
    const int first = wave * per, end = first + per < KT ? first + per : KT;
    const int64_t a_ks = p.a_ks ? p.a_ks : 128, b_ks = p.b_ks ? p.b_ks : 128;
    const int bn = p.N - n0;  // rows past a matrix repeat its last one; never stored
    uint8_t *const mine = smem + wave * (U * skinny_stage_bytes(MT));
    uint32_t *const my_scales = (uint32_t *)(smem + SKINNY_WAVES * U * skinny_stage_bytes(MT)) + wave * (U * 16 * MT);  // activations
    const uint32_t copy_to = __builtin_amdgcn_readfirstlane(lds_addr(mine));
    uint32_t a_voff[2 * MT], b_voff[2];
    auto chunk_of = [&](int row) { return (uint32_t)(((lane & 7) ^ swz_a(row)) << 4); };
#pragma unroll
    for (int q = 0; q < 2 * MT && SRC == SRC_CODES; q++) {
        const int row = 8 * q + (lane >> 3);
        a_voff[q] = (uint32_t)((row < p.M ? row : p.M - 1) * p.lda) + chunk_of(row);
    }
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const int row = 8 * q + (lane >> 3);
        b_voff[q] = (uint32_t)((row < bn ? row : bn - 1) * p.ldb) + chunk_of(row);
    }
    const uint8_t *const a_base = p.aq, *const b_base = p.bq + (int64_t)n0 * p.ldb;
    // scale words: lane l holds those of A row l (and row 64 + l) and of B row l % 16
    constexpr int SW = (MT * 16 + 63) / 64;
    const uint8_t *sa_at[SW];
#pragma unroll
    for (int w = 0; w < SW && SRC == SRC_CODES; w++) sa_at[w] = p.as + (int64_t)(64 * w + lane < p.M ? 64 * w + lane : p.M - 1) * p.ldas;
    const uint8_t *const sb_at = p.bs + (int64_t)(n0 + (r16 < bn ? r16 : bn - 1)) * p.ldbs;

    v4f acc[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) acc[i] = v4f{0.f, 0.f, 0.f, 0.f};
    for (int s0 = first; s0 < end; s0 += U) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the fragments of the previous pass are out of LDS
        uint32_t sa[U][SW], sb[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int s = s0 + u < end ? s0 + u : s0;  // an absent stage repeats the first one; never multiplied
#pragma unroll
            for (int w = 0; w < SW && SRC == SRC_CODES; w++) sa[u][w] = *(const uint32_t *)(sa_at[w] + 4 * s);
            sb[u] = *(const uint32_t *)(sb_at + 4 * s);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (s0 + u >= end) break;
            const uint8_t *const ga = uniform_ptr(a_base + (s0 + u) * a_ks), *const gb = uniform_ptr(b_base + (s0 + u) * b_ks);
            const uint32_t to = copy_to + u * skinny_stage_bytes(MT);
#pragma unroll
            for (int q = 0; q < 2; q++) dma16(gb, b_voff[q], to + (2 * MT + q) * 1024);
            if constexpr (SRC == SRC_CODES) {
#pragma unroll
                for (int q = 0; q < 2 * MT; q++) dma16(ga, a_voff[q], to + q * 1024);
            }
        }
        if constexpr (SRC != SRC_CODES) {
            typedef Elem<SRC> E;
            typename E::raw x[U][4 * MT];
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int q = 0; q < 4 * MT; q++) {
                    const int s = s0 + u < end ? s0 + u : s0, row = 4 * q + g < p.M ? 4 * q + g : p.M - 1;
                    x[u][q] = E::load_raw((const typename E::type *)p.aq + (int64_t)row * p.lda + 128 * s + 8 * r16);
                }
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int q = 0; q < 4 * MT; q++) {
                    if (4 * q >= p.M) break;  // rows past the matrix are multiplied as they lie in LDS and never stored
                    float v[8];
                    E::unpack(x[u][q], v);
                    if constexpr (SRC == MX_FP32) round_values<CAST>(v);
                    const uint32_t byte = scale_byte(quad_max(amax8(v)));
                    const float scale = block_scale(byte);
                    v2i codes;
                    codes[0] = (int)pack4_e4m3(v[0], v[1], v[2], v[3], scale);
                    codes[1] = (int)pack4_e4m3(v[4], v[5], v[6], v[7], scale);
                    const int row = 4 * q + g;
                    *(v2i *)(mine + u * skinny_stage_bytes(MT) + row * 128 + (((r16 >> 1) ^ swz_a(row)) << 4) + 8 * (r16 & 1)) = codes;
                    if ((r16 & 3) == 0) ((uint8_t *)(my_scales + u * 16 * MT + row))[r16 >> 2] = (uint8_t)byte;
                }
        }
        wait_vm_allow_c<0>();
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (s0 + u >= end) break;
            const uint8_t *const at = mine + u * skinny_stage_bytes(MT);
            auto fragment = [&](int row) {
                const int chunk = (g ^ swz_a(row)) << 4;
                const v4i lo = *(const v4i *)(at + row * 128 + chunk), hi = *(const v4i *)(at + row * 128 + (chunk ^ 64));
                return (v8i)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            };
            const v8i b = fragment(16 * MT + r16);
            const int bs = (int)(sb[u] >> (8 * g));
#pragma unroll
            for (int i = 0; i < MT; i++) {
                const uint32_t word = SRC == SRC_CODES ? (uint32_t)__shfl((int)sa[u][i / 4], 16 * (i % 4) + r16, 64) : my_scales[u * 16 * MT + 16 * i + r16];
                const int as = (int)(word >> (8 * g));
                acc[i] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fragment(16 * i + r16), b, acc[i], 0, 0, 0, as, 0, bs);
            }
        }
    }
    v4f *const red = (v4f *)smem;
    __syncthreads();  // every wave is done with its stages: the sums go over them
#pragma unroll
    for (int i = 0; i < MT; i++) red[(wave * MT + i) * 64 + lane] = acc[i];
    __syncthreads();
    if (wave >= MT) return;
    v4f sum = red[wave * 64 + lane];  // wave i adds and stores sub-tile i
#pragma unroll
    for (int w = 1; w < SKINNY_WAVES; w++) sum += red[(w * MT + wave) * 64 + lane];
    const int n = n0 + r16;
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int m = 16 * wave + 4 * g + v;
        if (m >= p.M || n >= p.N) continue;
        const int64_t at = (int64_t)m * p.ldc + n;
        if (CDT == MX_FP32) ((float *)p.c)[at] = sum[v];
        else if (CDT == MX_BF16) ((uint16_t *)p.c)[at] = (uint16_t)pack2_bf16(sum[v], 0.f);
        else ((_Float16 *)p.c)[at] = (_Float16)sum[v];
    }
}

}  // namespace mx
