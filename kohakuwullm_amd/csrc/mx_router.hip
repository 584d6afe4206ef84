// Top-k router of the mixture-of-experts block, for gfx950: scores, selection, gate weights and the histogram of the
// picks from one pass over the hidden states, and the backward of the gate weights into the hidden states and the router
// matrix.  Semantics: TopKRouter.route of the reference (src/kohakuwullm/models/components/moe.py:97-199) with sigmoid
// scores and one expert group.
//
// As a composition of library operators the same work is 15 launches forward and 20 backward over tensors of a few KB to
// a few MB, with the hidden states widened to fp32 in memory first: 160 + 300 us of a 1.55 ms block at 16384 tokens of
// 1024 and 64 experts, and nothing but launches at a few tokens.  Here it is two launches forward (25 us; one where the
// tokens fit a workgroup, which then needs no histogram cleared in front of it) and three backward (45 us).
#include <atomic>
#include <type_traits>

#include "mx_common.h"

namespace mx {

// 1 / (1 + e^-l) with the correctly rounded division and the library exponential: the selection compares these values,
// so they are kept as exact as fp32 gives them (unlike SwiGLU's sigmoid_f32).
__device__ __forceinline__ float router_sigmoid(float l) { return 1.0f / (1.0f + expf(-l)); }

// clamp(total, 1e-9) that keeps a NaN (fmaxf drops it: a token with one NaN score would get gates of 1e9 for its other picks)
__device__ __forceinline__ float clamp_total(float total) { return total < 1e-9f ? 1e-9f : total; }

// Unsigned integers in the order of the floats; NaN above everything, as torch.topk has it.
__device__ __forceinline__ uint32_t ordered_key(float f) {
    const uint32_t u = f2bits(f);
    if ((u & 0x7FFFFFFFu) > 0x7F800000u) return 0xFFFFFFFFu;
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// a raw element of a 16-bit or fp32 matrix that is not bf16
__device__ __forceinline__ float to_float(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }
__device__ __forceinline__ float to_float(float f) { return f; }

__device__ __forceinline__ float load_float(const void *p, int dtype, int64_t i) {
    if (dtype == MX_FP32) return ((const float *)p)[i];
    if (dtype == MX_BF16) return bits2f((uint32_t)((const uint16_t *)p)[i] << 16);
    return (float)((const _Float16 *)p)[i];
}

__device__ __forceinline__ void store_float(void *p, int dtype, int64_t i, float v) {
    if (dtype == MX_FP32) ((float *)p)[i] = v;
    else if (dtype == MX_BF16) ((uint16_t *)p)[i] = (uint16_t)f2bf16(v);
    else ((_Float16 *)p)[i] = (_Float16)v;
}

struct RouterArgs {
    const void *x;
    int64_t ldx;
    const void *w, *bias;
    int bias_dtype;
    int T, D, E, top_k, norm;
    float factor;
    int64_t *idx;
    void *weight;    // (T, top_k) in x's type
    float *scores;   // (T, top_k) fp32: the selected scores, what the backward needs; may be null
    int32_t *counts;
};

constexpr int ROUTER_WAVES = 8, ROUTER_ROWS = 16;

// Largest of the wave's 64 unsigned values, to every lane (DPP: a running maximum along the rows, then across them), for several
// values side by side.
template <int N>
__device__ __forceinline__ void wave_max_u32(uint32_t (&v)[N]) {
#define MX_DPP_MAX(ctrl, rows)                                                                          \
    _Pragma("unroll") for (int i = 0; i < N; i++) {                                                     \
        const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v[i], ctrl, rows, 0xF, false); \
        v[i] = v[i] > o ? v[i] : o;                                                                     \
    }
    MX_DPP_MAX(0x111, 0xF)  // row_shr:1
    MX_DPP_MAX(0x112, 0xF)
    MX_DPP_MAX(0x114, 0xF)
    MX_DPP_MAX(0x118, 0xF)
    MX_DPP_MAX(0x142, 0xA)  // row_bcast:15 into rows 1 and 3
    MX_DPP_MAX(0x143, 0xC)  // row_bcast:31 into rows 2 and 3
#undef MX_DPP_MAX
#pragma unroll
    for (int i = 0; i < N; i++) v[i] = (uint32_t)__builtin_amdgcn_readlane((int)v[i], 63);
}

template <int DT>
__device__ __forceinline__ v4f mfma_16bit(v4i a, v4i b, v4f c) {
    typedef __bf16 b8 __attribute__((ext_vector_type(8)));
    typedef _Float16 h8 __attribute__((ext_vector_type(8)));
    if constexpr (DT == MX_BF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, a), __builtin_bit_cast(b8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, a), __builtin_bit_cast(h8, b), c, 0, 0, 0);
}

// One workgroup: 16 MT tokens, all experts.  A lane's 16-byte load holds 8 consecutive K of one row of x (or of w), which is
// an operand of the 16-bit MFMA (16x16x32) as it stands; its products are exact and its sums fp32 (measured against fp64:
// rms error of a logit 2.4e-7 at D = 1024, the fp32 library product 3.9e-7).  Operands of mixed or fp32 type run on the fp32
// MFMA (16x16x4), step i taking element i of every lane.  The K axis is dealt to the eight waves 32 at a time, ROUTER_AHEAD
// such steps are requested before the first is used, and the waves' partial logits meet in LDS.
// Then a wave selects for two tokens, or for four at a time: top_k times the maximum of the experts' keys, one or more experts per
// lane; ties go to the lower expert.
// What bounds it: the loads of the operands at large token counts -- a lane group of 16 reads 16 rows, so a load instruction
// takes the texture path 64 clocks instead of 16 -- which is why a workgroup reads w once for 64 tokens when there are enough
// of them (16384 x 1024, 64 experts: 35 us with one tile of 16 tokens, 23 us with four; 26 with half as many loads in flight and
// one selection at a time), and the chain load - product - selection of one workgroup at small ones (9 us at 32 tokens).
constexpr int ROUTER_AHEAD = 4;
template <int XDT, int WDT, int NT, int MT>
__global__ __launch_bounds__(ROUTER_WAVES * 64, MT > 1 ? 2 : NT <= 8 ? 4 : 2) void router_topk_kernel(RouterArgs p) {
    typedef typename Elem<XDT>::type X;
    typedef typename Elem<WDT>::type W;
    constexpr int PITCH = NT * 16 + 4;
    constexpr int AHEAD = NT <= 4 && XDT != MX_FP32 && WDT != MX_FP32 ? ROUTER_AHEAD : 1;  // as registers allow
    extern __shared__ float slices[];  // [wave][token][expert], then the histogram
    int32_t *hist = (int32_t *)(slices + ROUTER_WAVES * ROUTER_ROWS * MT * PITCH);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
    const int first = blockIdx.x * ROUTER_ROWS * MT;
    for (int e = tid; e < p.E; e += ROUTER_WAVES * 64) hist[e] = 0;

    constexpr int Q = (NT * 16 + 63) / 64;  // experts per lane
    float bias[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) bias[q] = p.bias && lane + 64 * q < p.E ? load_float(p.bias, p.bias_dtype, lane + 64 * q) : 0.0f;

    const X *xr[MT];
    const W *wr[NT];
#pragma unroll
    for (int m = 0; m < MT; m++) {
        const int t = first + 16 * m + r;
        xr[m] = (const X *)p.x + (int64_t)(t < p.T ? t : p.T - 1) * p.ldx + 8 * g;
    }
#pragma unroll
    for (int j = 0; j < NT; j++) wr[j] = (const W *)p.w + (int64_t)(16 * j + r < p.E ? 16 * j + r : p.E - 1) * p.D + 8 * g;
    v4f acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[m][j] = v4f{0.f, 0.f, 0.f, 0.f};
    for (int kb = wave * 32; kb < p.D; kb += AHEAD * ROUTER_WAVES * 32) {
        typename Elem<XDT>::raw xa[AHEAD][MT];
        typename Elem<WDT>::raw b[AHEAD][NT];
#pragma unroll
        for (int s = 0; s < AHEAD; s++) {
            const int k0 = kb + s * ROUTER_WAVES * 32;
            const int k = k0 + 8 * g < p.D ? k0 : -8 * g;  // past the row: its start, and no use made of it (D % 8 == 0)
#pragma unroll
            for (int m = 0; m < MT; m++) xa[s][m] = Elem<XDT>::template load_raw<false>(xr[m] + k);
#pragma unroll
            for (int j = 0; j < NT; j++) b[s][j] = Elem<WDT>::template load_raw<false>(wr[j] + k);
        }
        __builtin_amdgcn_sched_barrier(0);  // all of them are requested before the first is waited for
#pragma unroll
        for (int s = 0; s < AHEAD; s++) {
            // past the end of a row both factors are zero (w may hold values that are not finite)
            const bool use = kb + s * ROUTER_WAVES * 32 + 8 * g < p.D;
            if constexpr (XDT == WDT && XDT != MX_FP32) {
                const v4i zero = {0, 0, 0, 0};
#pragma unroll
                for (int j = 0; j < NT; j++) {
                    const v4i bv = use ? __builtin_bit_cast(v4i, b[s][j]) : zero;
#pragma unroll
                    for (int m = 0; m < MT; m++)
                        acc[m][j] = mfma_16bit<XDT>(use ? __builtin_bit_cast(v4i, xa[s][m]) : zero, bv, acc[m][j]);
                }
            } else {
#pragma unroll
                for (int m = 0; m < MT; m++) {
                    float a[8];
                    Elem<XDT>::unpack(xa[s][m], a);
#pragma unroll
                    for (int j = 0; j < NT; j++) {
                        float bj[8];
                        Elem<WDT>::unpack(b[s][j], bj);
#pragma unroll
                        for (int i = 0; i < 8; i++)
                            acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(use ? a[i] : 0.0f, use ? bj[i] : 0.0f, acc[m][j], 0, 0, 0);
                    }
                }
            }
        }
    }
    float *mine = slices + wave * ROUTER_ROWS * MT * PITCH;
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) mine[(16 * m + 4 * g + v) * PITCH + 16 * j + r] = acc[m][j][v];
    __syncthreads();

    // A wave's tokens in groups of two or four side by side: every step of a selection waits for the one before it.  One barrier
    // for all tiles of 16: behind the stores of a tile's results, each further one waited for those to reach memory.
    constexpr int TOKENS = ROUTER_ROWS * MT / ROUTER_WAVES, U = TOKENS < 4 ? TOKENS : 4;
#pragma unroll 1
    for (int row0 = wave * TOKENS; row0 < (wave + 1) * TOKENS && first + row0 < p.T; row0 += U) {
        float score[U][Q];
        uint32_t key[U][Q];  // 0: no expert, or one already taken (no float has that key)
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const int e = lane + 64 * q;
            float part[U][ROUTER_WAVES];
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int s = 0; s < ROUTER_WAVES; s++) part[u][s] = slices[(s * ROUTER_ROWS * MT + row0 + u) * PITCH + (e < p.E ? e : 0)];
#pragma unroll
            for (int u = 0; u < U; u++) {
                float logit = 0.0f;
#pragma unroll
                for (int s = 0; s < ROUTER_WAVES; s++) logit += part[u][s];
                score[u][q] = router_sigmoid(logit);
                key[u][q] = e < p.E ? ordered_key(p.bias ? score[u][q] + bias[q] : score[u][q]) : 0u;
            }
        }
        float total[U], mine_s[U];
        int mine_e[U];
#pragma unroll
        for (int u = 0; u < U; u++) total[u] = mine_s[u] = 0.0f, mine_e[u] = 0;
        for (int i = 0; i < p.top_k; i++) {
            uint32_t best[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                best[u] = key[u][0];
#pragma unroll
                for (int q = 1; q < Q; q++) best[u] = key[u][q] > best[u] ? key[u][q] : best[u];
            }
            wave_max_u32(best);
#pragma unroll
            for (int u = 0; u < U; u++) {
                bool open = true;
#pragma unroll
                for (int q = 0; q < Q; q++) {
                    const uint64_t holders = __ballot(open && key[u][q] == best[u]);
                    if (Q > 1 && holders == 0) continue;  // uniform; at q the first lane of the lowest experts wins
                    const int at = __builtin_ctzll(holders);
                    const float s = bits2f((uint32_t)__builtin_amdgcn_readlane((int)f2bits(score[u][q]), at));
                    total[u] += s;
                    if (lane == i) mine_s[u] = s, mine_e[u] = at + 64 * q;
                    if (lane == at) key[u][q] = 0u;
                    open = false;
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int t = first + row0 + u;
            if (t >= p.T || lane >= p.top_k) continue;
            const float sum = clamp_total(total[u]);
            const int64_t at = (int64_t)t * p.top_k + lane;
            p.idx[at] = mine_e[u];
            store_float(p.weight, XDT, at, (p.norm ? mine_s[u] / sum : mine_s[u]) * p.factor);
            if (p.scores) p.scores[at] = mine_s[u];
            atomicAdd(&hist[mine_e[u]], 1);
        }
    }
    __syncthreads();
    for (int e = tid; e < p.E; e += ROUTER_WAVES * 64) {
        if (gridDim.x == 1) p.counts[e] = hist[e];  // the only workgroup: nothing was cleared for it
        else if (hist[e]) atomicAdd(&p.counts[e], hist[e]);
    }
}

__global__ __launch_bounds__(256) void router_clear_kernel(int32_t *counts, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) counts[i] = 0;
}

struct RouterBwdArgs {
    const void *gw;  // upstream gradient of the gate weights, (T, top_k)
    int gw_dtype;
    const int64_t *idx;
    const float *scores;
    const void *x;
    int64_t ldx;
    const void *w;
    int T, D, E, top_k, norm;
    float factor;
    void *dx;
    int64_t lddx;
    const void *onto;  // added to dx before it is rounded, in x's type, or null
    int64_t ldonto;
    float *partial;  // [chunk][E][D]: dW of `chunk_tokens` tokens each
    int chunks, chunk_tokens;
};

// d loss / d logit of a pick, through the factor (in g already), the optional normalisation and the sigmoid: w_i = f s_i / S with
// S = sum s (or 1) gives ds_i = f (g_i - [S above the clamp] (sum_j g_j s_j) / S) / S.
__device__ __forceinline__ float pick_gradient(const RouterBwdArgs &p, float g, float s, float sum, float dot) {
    float ds = g;
    if (p.norm) {
        const float S = clamp_total(sum);
        ds = (g - (sum < 1e-9f ? 0.0f : dot / S)) / S;
    }
    return ds * s * (1.0f - s);
}

template <int XDT>
__device__ __forceinline__ void dx_store(const RouterBwdArgs &p, int64_t t, int col, const float (&acc)[8]) {
    typename Elem<XDT>::type *dst = (typename Elem<XDT>::type *)p.dx + t * p.lddx + col;
    if (XDT == MX_FP32) {
        ((v4f *)dst)[0] = v4f{acc[0], acc[1], acc[2], acc[3]};
        ((v4f *)dst)[1] = v4f{acc[4], acc[5], acc[6], acc[7]};
    } else if (XDT == MX_BF16) {
        *(v4i *)dst = v4i{(int)pack2_bf16(acc[0], acc[1]), (int)pack2_bf16(acc[2], acc[3]), (int)pack2_bf16(acc[4], acc[5]),
                          (int)pack2_bf16(acc[6], acc[7])};
    } else {
        typedef _Float16 h8 __attribute__((ext_vector_type(8)));
        h8 h;
#pragma unroll
        for (int c = 0; c < 8; c++) h[c] = (_Float16)acc[c];
        *(h8 *)dst = h;
    }
}

// dx[t] = sum over the picks of dlogit * w[expert], a wave per token.  top_k of E terms are not zero, so this is a gather of
// top_k rows of the router matrix, not a matrix product.  Where the caller has a gradient of the same hidden states in hand (what
// the experts give), the sums start from it: a launch and a pass over three matrices less.
// pick(i) gives the gradient and the expert of the token's pick i, the same ones to every lane.
template <int XDT, int WDT, typename F>
__device__ __forceinline__ void router_dx_row(const RouterBwdArgs &p, int64_t t, int lane, F &&pick) {
    typedef typename Elem<XDT>::type X;
    typedef typename Elem<WDT>::type W;
    for (int first = 0; first < p.D; first += 512) {  // every lane of the wave goes along: the picks are read from them
        const int col = first + lane * 8, from = col < p.D ? col : 0;
        typename Elem<XDT>::raw below;
        if (p.onto) below = Elem<XDT>::template load_raw<false>((const X *)p.onto + t * p.ldonto + from);
        float acc[8];
        for (int i0 = 0; i0 < p.top_k; i0 += 8) {
            typename Elem<WDT>::raw row[8];
            float dl[8];
#pragma unroll
            for (int i = 0; i < 8; i++)  // all of them are requested before the first is waited for
                if (i0 + i < p.top_k) {
                    int e;
                    pick(i0 + i, dl[i], e);
                    row[i] = Elem<WDT>::template load_raw<false>((const W *)p.w + (int64_t)e * p.D + from);
                }
            if (i0 == 0) {
                if (p.onto) {
                    Elem<XDT>::unpack(below, acc);
                } else {
#pragma unroll
                    for (int c = 0; c < 8; c++) acc[c] = 0.0f;
                }
            }
#pragma unroll
            for (int i = 0; i < 8; i++) {
                if (i0 + i >= p.top_k) break;  // uniform
                float wv[8];
                Elem<WDT>::unpack(row[i], wv);
#pragma unroll
                for (int c = 0; c < 8; c++) acc[c] += dl[i] * wv[c];
            }
        }
        if (col < p.D) dx_store<XDT>(p, t, col, acc);
    }
}

// The picks' gradients in two ways, with the same sums in the same order (launch_router_dx chooses).
// Few tokens: lane i of a wave forms the gradient of the token's pick i, the sums over the picks go lane by lane through scalar
// registers, and the next token's picks are requested ahead.  A wave waits for nobody else, but all its lanes form six gradients.
constexpr int ROUTER_MAX_K = 16, ROUTER_DX_TOKENS = 16;
template <int XDT, int WDT>
__global__ __launch_bounds__(256) void router_dx_few_kernel(RouterBwdArgs p) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t stride = (int64_t)gridDim.x * 4, mine = lane < p.top_k ? lane : 0;
    int64_t t = (int64_t)blockIdx.x * 4 + wave;
    if (t >= p.T) return;
    struct Pick {
        float g, s;
        int e;
    };
    auto pick_of = [&](int64_t token) {
        const int64_t at = token * p.top_k + mine;
        return Pick{load_float(p.gw, p.gw_dtype, at) * p.factor, p.scores[at], (int)p.idx[at]};
    };
    Pick next = pick_of(t);
    for (; t < p.T; t += stride) {
        const float g = next.g, s = next.s;
        const int mine_e = next.e;
        next = pick_of(t + stride < p.T ? t + stride : t);
        float sum = 0.0f, dot = 0.0f;
        if (p.norm) {
            for (int j = 0; j < p.top_k; j++) {
                const float sj = bits2f((uint32_t)__builtin_amdgcn_readlane((int)f2bits(s), j));
                sum += sj;
                dot += bits2f((uint32_t)__builtin_amdgcn_readlane((int)f2bits(g), j)) * sj;
            }
        }
        const float mine_dl = pick_gradient(p, g, s, sum, dot);
        router_dx_row<XDT, WDT>(p, t, lane, [&](int i, float &dl, int &e) {
            dl = bits2f((uint32_t)__builtin_amdgcn_readlane((int)f2bits(mine_dl), i));
            e = __builtin_amdgcn_readlane(mine_e, i);
        });
    }
}

// Many tokens: a workgroup forms the gradients of sixteen tokens' picks in LDS, a thread per pick, behind two round trips to memory
// and two barriers, which other workgroups fill; its waves then gather four tokens each.
template <int XDT, int WDT, bool ONTO>
__global__ __launch_bounds__(256) void router_dx_kernel(RouterBwdArgs p) {
    __shared__ v2i picks[ROUTER_DX_TOKENS * ROUTER_MAX_K];
    __shared__ v2f gs[ROUTER_DX_TOKENS * ROUTER_MAX_K];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t lo = (int64_t)blockIdx.x * ROUTER_DX_TOKENS;
    const int n = (int)(p.T - lo < ROUTER_DX_TOKENS ? p.T - lo : ROUTER_DX_TOKENS);
    static_assert(ROUTER_DX_TOKENS * ROUTER_MAX_K <= 256, "a pick per thread");
    const int mine = threadIdx.x, total = n * p.top_k;
    float g = 0.0f, s = 0.0f;
    int expert = 0;
    if (mine < total) {
        const int64_t at = lo * p.top_k + mine;
        g = load_float(p.gw, p.gw_dtype, at) * p.factor, s = p.scores[at], expert = (int)p.idx[at];
        gs[mine] = v2f{g, s};
    }
    __syncthreads();
    if (mine < total) {
        float sum = 0.0f, dot = 0.0f;
        if (p.norm) {
            const int first = mine / p.top_k * p.top_k;
            for (int j = 0; j < p.top_k; j++) {
                const v2f other = gs[first + j];
                sum += other[1];
                dot += other[0] * other[1];
            }
        }
        picks[mine] = v2i{(int)f2bits(pick_gradient(p, g, s, sum, dot)), expert};
    }
    __syncthreads();
    for (int u = wave; u < n; u += 4) {
        if constexpr (ONTO) {  // requested together with the rows
            router_dx_row<XDT, WDT>(p, lo + u, lane, [&](int i, float &dl, int &e) {
                const v2i pick = picks[u * p.top_k + i];
                dl = bits2f((uint32_t)pick[0]), e = pick[1];
            });
        } else {
            for (int col = lane * 8; col < p.D; col += 512) {
                float acc[8];
#pragma unroll
                for (int c = 0; c < 8; c++) acc[c] = 0.0f;
#pragma unroll 4
                for (int i = 0; i < p.top_k; i++) {
                    const v2i pick = picks[u * p.top_k + i];
                    float wv[8];
                    Elem<WDT>::load8((const typename Elem<WDT>::type *)p.w + (int64_t)pick[1] * p.D + col, wv);
#pragma unroll
                    for (int c = 0; c < 8; c++) acc[c] += bits2f((uint32_t)pick[0]) * wv[c];
                }
                dx_store<XDT>(p, lo + u, col, acc);
            }
        }
    }
}

// dW[e] += dlogit[t, e] x[t]: a matrix product over the tokens.  A workgroup owns 64 experts, 256 columns (64 per wave) and
// a chunk of tokens; the gradients of the chunk stand dense in LDS, one row of tokens per expert, K-minor as the MFMA reads
// them.  A lane loads four columns of each of eight tokens, so column tile j of a wave holds columns c0 + 4 r + j.
// bf16 hidden states run on the bf16 MFMA: the fp32 gradient is kept whole as the sum of three bf16 (8 bits each), the
// products are exact and the sums fp32, and 48 MFMAs per 32 tokens take 768 clocks where the fp32 form needs 4096 (16384 x
// 1024, 64 experts: 22 us, 25 with four waves, one step of x ahead and the picks fetched in turn; the read of x and 17 MB of
// partial sums take 10 of them, the chain picks - gradients - products most of the others); other types take the fp32 MFMA.  The chunks' fp32 partial matrices are added in order by router_dw_kernel (deterministic).
constexpr int ROUTER_CHUNK = 256, ROUTER_DW_COLS = 256, ROUTER_DW_THREADS = 512;
__host__ __device__ constexpr int router_dw_pitch(int tokens, bool split) { return split ? tokens + 8 : tokens + 4; }
__host__ __device__ constexpr int router_dw_lds(int tokens, int top_k, bool split) {
    const int used = (split ? 3 * 64 * router_dw_pitch(tokens, true) * 2 : 64 * router_dw_pitch(tokens, false) * 4) + tokens * top_k * 8;
    return used < 65536 ? 65536 : used;  // at the end the odd steps' sums of 64 x 256 elements
}
// f(std::integral_constant<int, 0>{}), ..., f(std::integral_constant<int, N - 1>{})
template <int N, int I = 0, typename F>
__device__ __forceinline__ void static_for_steps(F &&f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for_steps<N, I + 1>(f);
    }
}

template <int XDT>
__global__ __launch_bounds__(ROUTER_DW_THREADS) void router_dw_partial_kernel(RouterBwdArgs p) {
    typedef typename Elem<XDT>::type X;
    constexpr bool SPLIT = XDT == MX_BF16;
    typedef X x4 __attribute__((ext_vector_type(4)));
    extern __shared__ __attribute__((aligned(16))) uint8_t dw_smem[];
    const int pitch = router_dw_pitch(p.chunk_tokens, SPLIT);  // elements
    const int plane = 64 * pitch;
    const int dense_bytes = SPLIT ? 3 * plane * 2 : plane * 4;
    v2f *const gs = (v2f *)(dw_smem + dense_bytes);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
    const int e0 = (int)blockIdx.y * 64, col = (int)blockIdx.x * ROUTER_DW_COLS + (wave & 3) * 64 + 4 * r;
    const int half = wave >> 2;  // waves 0-3 take the even steps of 32 tokens, waves 4-7 the odd ones
    const int64_t lo = (int64_t)blockIdx.z * p.chunk_tokens;
    const int n = (int)(p.T - lo < p.chunk_tokens ? p.T - lo : p.chunk_tokens);
    const bool col_in = col < p.D;
    const X *const base = (const X *)p.x + lo * p.ldx + (col_in ? col : 0);
    auto load = [&](int step, x4 (&raw)[8]) {  // tokens 32 step + 8 g + i, the last one again past the end (its gradient is 0)
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int t = 32 * step + 8 * g + i;
            raw[i] = *(const x4 *)(base + (int64_t)(t < n ? t : n - 1) * p.ldx);
        }
    };
    // The chunk's picks, one thread per pick and all of them requested at once, in front of x: loads return in order.
    constexpr int PICKS = ROUTER_CHUNK * ROUTER_MAX_K / ROUTER_DW_THREADS;
    const int total = n * p.top_k;
    float pg[PICKS], ps[PICKS];
    int pe[PICKS];
#pragma unroll
    for (int k = 0; k < PICKS; k++) {
        const int i = tid + k * ROUTER_DW_THREADS;
        if (k * ROUTER_DW_THREADS >= total) break;  // uniform
        const int64_t at = lo * p.top_k + (i < total ? i : 0);
        pg[k] = load_float(p.gw, p.gw_dtype, at) * p.factor, ps[k] = p.scores[at], pe[k] = (int)p.idx[at];
    }
    constexpr int AHEAD = 4;  // of the wave's steps
    const int steps = (n + 31) / 32;
    x4 buf[AHEAD][8];
    static_for_steps<AHEAD>([&](auto s) {
        if (2 * s.value + half < steps) load(2 * s.value + half, buf[s.value]);
    });
    for (int i = tid * 16; i < dense_bytes; i += ROUTER_DW_THREADS * 16) *(v4i *)(dw_smem + i) = v4i{0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < PICKS; k++) {
        const int i = tid + k * ROUTER_DW_THREADS;
        if (i < total) gs[i] = v2f{pg[k], ps[k]};
    }
    __syncthreads();  // the zeros are in place as well
#pragma unroll
    for (int k = 0; k < PICKS; k++) {
        const int i = tid + k * ROUTER_DW_THREADS;
        if (k * ROUTER_DW_THREADS >= total) break;
        if (i >= total) continue;
        float sum = 0.0f, dot = 0.0f;
        if (p.norm) {
            const int token0 = i / p.top_k * p.top_k;
            for (int j = 0; j < p.top_k; j++) {
                const v2f other = gs[token0 + j];
                sum += other[1];
                dot += other[0] * other[1];
            }
        }
        const float v = pick_gradient(p, pg[k], ps[k], sum, dot);
        const int e = pe[k] - e0, at = e * pitch + i / p.top_k;
        if (e < 0 || e >= 64) continue;
        if constexpr (SPLIT) {
            uint16_t *d = (uint16_t *)dw_smem;
            const uint32_t hi = f2bf16(v);
            const float rest = v - bits2f(hi << 16);
            const uint32_t mid = f2bf16(rest);
            d[at] = (uint16_t)hi;
            d[plane + at] = (uint16_t)mid;
            d[2 * plane + at] = (uint16_t)f2bf16(rest - bits2f(mid << 16));
        } else {
            ((float *)dw_smem)[at] = v;
        }
    }
    __syncthreads();
    v4f acc[4][4];
#pragma unroll
    for (int m = 0; m < 4; m++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[m][j] = v4f{0.f, 0.f, 0.f, 0.f};
    auto use = [&](int step, const x4 (&cur)[8]) {
        const int tok = 32 * step + 8 * g;
        if constexpr (SPLIT) {
            v4i b[4];
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) b[j][q] = (int)((uint32_t)cur[2 * q][j] | (uint32_t)cur[2 * q + 1][j] << 16);
#pragma unroll
            for (int m = 0; m < 4; m++) {
                v4i a[3];
#pragma unroll
                for (int h = 0; h < 3; h++) a[h] = *(const v4i *)((const uint16_t *)dw_smem + h * plane + (16 * m + r) * pitch + tok);
#pragma unroll
                for (int j = 0; j < 4; j++)
#pragma unroll
                    for (int h = 2; h >= 0; h--) acc[m][j] = mfma_16bit<MX_BF16>(a[h], b[j], acc[m][j]);
            }
        } else {
#pragma unroll
            for (int m = 0; m < 4; m++) {
                const v4f *src = (const v4f *)((const float *)dw_smem + (16 * m + r) * pitch + tok);
                const v4f a0 = src[0], a1 = src[1];
#pragma unroll
                for (int i = 0; i < 8; i++)
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(i < 4 ? a0[i & 3] : a1[i & 3], to_float(cur[i][j]), acc[m][j], 0, 0, 0);
            }
        }
    };
    for (int first = half; first < steps; first += 2 * AHEAD)
        static_for_steps<AHEAD>([&](auto s) {
            const int step = first + 2 * s.value;
            if (step >= steps) return;
            use(step, buf[s.value]);
            if (step + 2 * AHEAD < steps) load(step + 2 * AHEAD, buf[s.value]);
        });
    __syncthreads();  // the gradients have been read: their place takes the odd steps' sums
    v4f *const odd = (v4f *)dw_smem + (wave & 3) * 16 * 64 + lane;
    if (half) {
#pragma unroll
        for (int i = 0; i < 16; i++) odd[i * 64] = acc[i >> 2][i & 3];
    }
    __syncthreads();
    if (half) return;
#pragma unroll
    for (int i = 0; i < 16; i++) acc[i >> 2][i & 3] += odd[i * 64];
    if (!col_in) return;
#pragma unroll
    for (int m = 0; m < 4; m++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int e = e0 + 16 * m + 4 * g + v;
            if (e < p.E)
                *(v4f *)(p.partial + ((int64_t)blockIdx.z * p.E + e) * p.D + col) = v4f{acc[m][0][v], acc[m][1][v], acc[m][2][v], acc[m][3][v]};
        }
}

// dW = the sum of the chunks' partial matrices in the router matrix's type.  A workgroup takes 256 elements, its four waves
// a quarter of the chunks each (every fourth), and the quarters are added in order: the same sum on every run.
template <int WDT>
__global__ __launch_bounds__(256) void router_dw_kernel(const float *__restrict__ partial, int chunks, int64_t n, void *__restrict__ dw) {
    __shared__ v4f quarter[3][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t i = ((int64_t)blockIdx.x * 64 + lane) * 4;
    v4f s = v4f{0.f, 0.f, 0.f, 0.f};
    if (i < n) {
#pragma unroll 4
        for (int c = wave; c < chunks; c += 4) s += *(const v4f *)(partial + c * n + i);
    }
    if (wave) quarter[wave - 1][lane] = s;
    __syncthreads();
    if (wave || i >= n) return;
#pragma unroll
    for (int w = 0; w < 3; w++) s += quarter[w][lane];
#pragma unroll
    for (int v = 0; v < 4; v++) store_float(dw, WDT, i + v, s[v]);
}

static bool router_aligned(const void *p) { return ((uintptr_t)p & 15) == 0; }

static bool router_shape_ok(int x_dtype, int w_dtype, int64_t ldx, int64_t T, int64_t D, int64_t E, int64_t top_k) {
    const bool x_ok = x_dtype == MX_BF16 || x_dtype == MX_FP16 || x_dtype == MX_FP32;
    return x_ok && (w_dtype == x_dtype || w_dtype == MX_FP32) && T >= 0 && T < 0x7FFFFFFF / 16 && D > 0 && D < (1 << 24) && E > 0 &&
           top_k > 0 && top_k <= E && ldx >= D;
}

// Tokens per partial dW matrix: a workgroup for every CU (column blocks x expert groups of them per chunk), in whole
// steps of 32, at most ROUTER_CHUNK (the dense gradients of a chunk stand in LDS).
static int router_chunk_tokens(int64_t T, int64_t D, int64_t E, int cus) {
    const int64_t per_chunk = ((D + ROUTER_DW_COLS - 1) / ROUTER_DW_COLS) * ((E + 63) / 64);
    const int64_t tokens = ((T * per_chunk + cus - 1) / cus + 31) / 32 * 32;
    return (int)(tokens < 32 ? 32 : tokens > ROUTER_CHUNK ? ROUTER_CHUNK : tokens);
}

template <int XDT, int WDT, int NT, int MT>
static int launch_router(const RouterArgs &a, hipStream_t st) {
    const int lds = ROUTER_WAVES * ROUTER_ROWS * MT * (NT * 16 + 4) * 4 + NT * 16 * 4;
    if (lds > 65536) {
        static std::atomic<uint64_t> done;
        if (!allow_dynamic_lds((const void *)router_topk_kernel<XDT, WDT, NT, MT>, lds, done)) return MX_ELAUNCH;
    }
    const unsigned blocks = (unsigned)((a.T + ROUTER_ROWS * MT - 1) / (ROUTER_ROWS * MT));
    if (blocks != 1) router_clear_kernel<<<dim3((a.E + 255) / 256), dim3(256), 0, st>>>(a.counts, a.E);
    if (blocks) router_topk_kernel<XDT, WDT, NT, MT><<<dim3(blocks), dim3(ROUTER_WAVES * 64), lds, st>>>(a);
    return hipGetLastError() == hipSuccess ? MX_OK : MX_ELAUNCH;
}

// More rows of x per read of w once that leaves a workgroup for every CU (see the kernel).
template <int XDT, int WDT, int NT>
static int launch_router_mt(const RouterArgs &a, hipStream_t st) {
    if constexpr (NT <= 4 && XDT == WDT && XDT != MX_FP32) {
        const int64_t rows = (int64_t)ROUTER_ROWS * num_cus();
        if (a.T >= 3 * rows) return launch_router<XDT, WDT, NT, 4>(a, st);
        if (a.T > rows) return launch_router<XDT, WDT, NT, 2>(a, st);
    }
    return launch_router<XDT, WDT, NT, 1>(a, st);
}

template <int XDT, int WDT>
static int launch_router_nt(const RouterArgs &a, hipStream_t st) {
    if (a.E <= 16) return launch_router_mt<XDT, WDT, 1>(a, st);
    if (a.E <= 32) return launch_router_mt<XDT, WDT, 2>(a, st);
    if (a.E <= 64) return launch_router_mt<XDT, WDT, 4>(a, st);
    if (a.E <= 128) return launch_router_mt<XDT, WDT, 8>(a, st);
    return launch_router_mt<XDT, WDT, 16>(a, st);
}

// Which of the two kernels: what a wave waits for decides while the chip is not full, and the instructions per token afterwards.
// us few / many, bf16:
//   tokens   1024, 6 picks   2048, 6    1024, 16    4096, 8     512, 6     256, 4     1024, 6 onto a gradient
//   2777       5.6 / 9.7    8.5 / 16.7  8.5 / 13.3   15 / 27   4.4 / 5.8  4.4 / 4.2     5.9 / 10.2
//   8192      10.3 / 11.8  16.7 / 20.4 17.2 / 16.6   30 / 34   7.1 / 7.1  6.0 / 4.8    11.9 / 14.0
//   12288     13.1 / 13.1  21.8 / 23.6 22.9 / 20.2   41 / 42   9.2 / 8.1  7.4 / 5.4    19.4 / 19.3
//   16384     17.0 / 15.1  26.7 / 26.6 30.4 / 24.6   56 / 53  11.6 / 9.1  9.4 / 6.2    26.2 / 22.9
//   65536     54.4 / 39.1                106 / 78             36.6 / 23   30 / 16      100 / 90
static bool dx_few(const RouterBwdArgs &a) { return a.T <= (a.D <= 512 ? 32 : 48) * num_cus(); }

template <int XDT, int WDT>
static void launch_router_dx(const RouterBwdArgs &a, hipStream_t st) {
    const int64_t tokens = dx_few(a) ? 4 : ROUTER_DX_TOKENS, blocks = (a.T + tokens - 1) / tokens, most = 8 * (int64_t)num_cus();
    const dim3 grid((unsigned)(dx_few(a) && blocks > most ? most : blocks)), block(256);  // few: 32 waves per CU, in strides
    if (dx_few(a)) router_dx_few_kernel<XDT, WDT><<<grid, block, 0, st>>>(a);
    else if (a.onto) router_dx_kernel<XDT, WDT, true><<<grid, block, 0, st>>>(a);
    else router_dx_kernel<XDT, WDT, false><<<grid, block, 0, st>>>(a);
}

template <int XDT>
static int launch_router_dw(const RouterBwdArgs &a, hipStream_t st) {
    static std::atomic<uint64_t> done;
    const int most = router_dw_lds(ROUTER_CHUNK, ROUTER_MAX_K, XDT == MX_BF16);
    static_assert(router_dw_lds(ROUTER_CHUNK, ROUTER_MAX_K, true) <= 160 * 1024, "gradients and picks of a chunk fit the LDS");
    if (!allow_dynamic_lds((const void *)router_dw_partial_kernel<XDT>, most < 65536 ? 65536 : most, done)) return MX_ELAUNCH;
    const dim3 grid((unsigned)((a.D + ROUTER_DW_COLS - 1) / ROUTER_DW_COLS), (unsigned)((a.E + 63) / 64), (unsigned)a.chunks);
    router_dw_partial_kernel<XDT><<<grid, dim3(ROUTER_DW_THREADS), router_dw_lds(a.chunk_tokens, a.top_k, XDT == MX_BF16), st>>>(a);
    return MX_OK;
}

}  // namespace mx

using namespace mx;

extern "C" int mx_router_topk(const void *x, int x_dtype, int64_t ldx, const void *w, int w_dtype, const void *bias,
                              int bias_dtype, int64_t T, int64_t D, int64_t E, int64_t top_k, int norm, float factor,
                              int64_t *idx, void *weight, float *scores, int32_t *counts, void *stream) {
    if (!router_shape_ok(x_dtype, w_dtype, ldx, T, D, E, top_k) || !counts || !w || (T > 0 && (!x || !idx || !weight))) return MX_EINVAL;
    if (bias && bias_dtype != MX_BF16 && bias_dtype != MX_FP16 && bias_dtype != MX_FP32) return MX_EINVAL;
    const int xs = x_dtype == MX_FP32 ? 4 : 2;
    if (D % 8 || E > 256 || top_k > 64 || !router_aligned(x) || !router_aligned(w) || (ldx * xs) % 16) return MX_EUNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    if (stream_is_capturing(st)) return MX_ECAPTURE;
    const RouterArgs a = {x, ldx, w, bias, bias_dtype, (int)T, (int)D, (int)E, (int)top_k, norm != 0, factor, idx, weight, scores, counts};
    if (x_dtype == MX_BF16) return w_dtype == MX_FP32 ? launch_router_nt<MX_BF16, MX_FP32>(a, st) : launch_router_nt<MX_BF16, MX_BF16>(a, st);
    if (x_dtype == MX_FP16) return w_dtype == MX_FP32 ? launch_router_nt<MX_FP16, MX_FP32>(a, st) : launch_router_nt<MX_FP16, MX_FP16>(a, st);
    return launch_router_nt<MX_FP32, MX_FP32>(a, st);
}

extern "C" int64_t mx_router_backward_workspace(int64_t T, int64_t D, int64_t E) {
    if (T < 0 || D <= 0 || E <= 0) return -1;
    const int64_t tokens = router_chunk_tokens(T, D, E, num_cus());
    const int64_t chunks = T ? (T + tokens - 1) / tokens : 1;
    return chunks * E * D;
}

extern "C" int mx_router_topk_backward(const void *grad_weight, int gw_dtype, const int64_t *idx, const float *scores,
                                       const void *x, int x_dtype, int64_t ldx, const void *w, int w_dtype, int64_t T,
                                       int64_t D, int64_t E, int64_t top_k, int norm, float factor, void *dx, int64_t lddx,
                                       void *dw, float *workspace, int64_t workspace_len, void *stream) {
    return mx_router_topk_backward_onto(nullptr, 0, grad_weight, gw_dtype, idx, scores, x, x_dtype, ldx, w, w_dtype, T, D, E, top_k, norm, factor,
                                        dx, lddx, dw, workspace, workspace_len, stream);
}

extern "C" int mx_router_topk_backward_onto(const void *onto, int64_t ldonto, const void *grad_weight, int gw_dtype, const int64_t *idx,
                                            const float *scores, const void *x, int x_dtype, int64_t ldx, const void *w, int w_dtype, int64_t T,
                                            int64_t D, int64_t E, int64_t top_k, int norm, float factor, void *dx, int64_t lddx,
                                            void *dw, float *workspace, int64_t workspace_len, void *stream) {
    if (!router_shape_ok(x_dtype, w_dtype, ldx, T, D, E, top_k) || !w || (T > 0 && (!grad_weight || !idx || !scores || !x)) ||
        (gw_dtype != MX_BF16 && gw_dtype != MX_FP16 && gw_dtype != MX_FP32) || (dx && lddx < D) ||
        (onto && (!dx || ldonto < D)))
        return MX_EINVAL;
    if (dw && (!workspace || workspace_len < mx_router_backward_workspace(T, D, E))) return MX_EINVAL;
    const int xs = x_dtype == MX_FP32 ? 4 : 2;
    if (D % 8 || top_k > ROUTER_MAX_K || !router_aligned(x) || !router_aligned(w) || !router_aligned(dx) || !router_aligned(workspace) ||
        (ldx * xs) % 16 || (lddx * xs) % 16 || (onto && (!router_aligned(onto) || (ldonto * xs) % 16)))
        return MX_EUNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    if (stream_is_capturing(st)) return MX_ECAPTURE;
    RouterBwdArgs a = {grad_weight, gw_dtype, idx, scores, x, ldx, w, (int)T, (int)D, (int)E, (int)top_k, norm != 0, factor, dx, lddx, onto, ldonto, workspace,
                       0, 0};
    a.chunk_tokens = router_chunk_tokens(T, D, E, num_cus());
    a.chunks = T ? (int)((T + a.chunk_tokens - 1) / a.chunk_tokens) : 1;
    if (a.chunks > 65535) return MX_EUNSUPPORTED;
    if (dx && T) {
        if (x_dtype == MX_BF16 && w_dtype == MX_BF16) launch_router_dx<MX_BF16, MX_BF16>(a, st);
        else if (x_dtype == MX_BF16) launch_router_dx<MX_BF16, MX_FP32>(a, st);
        else if (x_dtype == MX_FP16 && w_dtype == MX_FP16) launch_router_dx<MX_FP16, MX_FP16>(a, st);
        else if (x_dtype == MX_FP16) launch_router_dx<MX_FP16, MX_FP32>(a, st);
        else launch_router_dx<MX_FP32, MX_FP32>(a, st);
    }
    if (dw) {
        const int rc = x_dtype == MX_BF16   ? launch_router_dw<MX_BF16>(a, st)
                       : x_dtype == MX_FP16 ? launch_router_dw<MX_FP16>(a, st)
                                            : launch_router_dw<MX_FP32>(a, st);
        if (rc != MX_OK) return rc;
    }
    if (dw) {
        const int64_t n = E * D;
        const dim3 grid((unsigned)((n / 4 + 63) / 64)), block(256);
        if (w_dtype == MX_BF16) router_dw_kernel<MX_BF16><<<grid, block, 0, st>>>(workspace, a.chunks, n, dw);
        else if (w_dtype == MX_FP16) router_dw_kernel<MX_FP16><<<grid, block, 0, st>>>(workspace, a.chunks, n, dw);
        else router_dw_kernel<MX_FP32><<<grid, block, 0, st>>>(workspace, a.chunks, n, dw);
    }
    return hipGetLastError() == hipSuccess ? MX_OK : MX_ELAUNCH;
}
