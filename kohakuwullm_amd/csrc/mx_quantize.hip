// MXFP8 quantizers for gfx950: row axis, column axis, both at once, and SwiGLU -> MXFP8.
//
// All of them are HBM-streaming kernels: 16-byte coalesced loads, per-32 amax by a
// DPP quad reduction (row axis) or an in-register + cross-lane reduction (column
// axis), the UE8M0 byte from the fp32 exponent/mantissa bits, an exact multiply by
// 2^-e, and the hardware RTNE e4m3 conversion.  Semantics follow _quantize_block of
// the reference (src/kohakuwullm/kernels/mxfp8/quantize.py:39-56).
#include "mx_common.h"

namespace mx {

// ------------------------------------------------------------------------------------
// Row axis.  One lane owns 8 consecutive elements; the 4 lanes of a quad own one block.
// ------------------------------------------------------------------------------------

// OR the quad's byte into a dword holding the 4 bytes of a 16-lane row, in block order.
__device__ __forceinline__ uint32_t gather_row_scales(uint32_t byte, int lane) {
    uint32_t v = byte << ((lane & 12) << 1);
    v |= (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x124, 0xF, 0xF, true);  // row_ror:4
    v |= (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x128, 0xF, 0xF, true);  // row_ror:8
    return v;
}

// CDT: the type fp32 values are rounded to before they are quantized (MX_FP32: none).
template <int DT, int U, bool FLAT, int CDT = MX_FP32>
__global__ __launch_bounds__(256) void quant_rows_kernel(const void *__restrict__ x, uint32_t chunks_per_row,
                                                          int64_t sx_row, uint8_t *__restrict__ q, int64_t ldq,
                                                          uint8_t *__restrict__ s, int64_t lds, uint32_t total_chunks,
                                                          int pack_scales) {
    typedef typename Elem<DT>::type T;
    const int lane = threadIdx.x & 63;
    const uint32_t base = blockIdx.x * (uint32_t)(U * 256) + threadIdx.x;
    float v[U][8];
    int64_t qoff[U], soff[U];
    bool ok[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        uint32_t chunk = base + u * 256;
        ok[u] = chunk < total_chunks;
        int64_t xoff;
        if (FLAT) {
            xoff = (int64_t)chunk * 8;
            qoff[u] = (int64_t)chunk * 8;
            soff[u] = chunk >> 2;
        } else {
            uint32_t row = chunk / chunks_per_row;
            uint32_t col = chunk - row * chunks_per_row;
            xoff = (int64_t)row * sx_row + (int64_t)col * 8;
            qoff[u] = (int64_t)row * ldq + (int64_t)col * 8;
            soff[u] = (int64_t)row * lds + (col >> 2);
        }
        if (ok[u]) {
            Elem<DT>::load8((const T *)x + xoff, v[u]);
            round_values<CDT>(v[u]);
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++) v[u][i] = 0.0f;
        }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
        float amax = quad_max(amax8(v[u]));
        uint32_t byte = scale_byte(amax);
        const float scale = block_scale(byte);
        uint32_t packed = gather_row_scales(byte, lane);
        if (ok[u]) {
            v2i codes;
            codes[0] = (int)pack4_e4m3(v[u][0], v[u][1], v[u][2], v[u][3], scale);
            codes[1] = (int)pack4_e4m3(v[u][4], v[u][5], v[u][6], v[u][7], scale);
            *(v2i *)(q + qoff[u]) = codes;
            // The 16 lanes of a DPP row hold 4 consecutive blocks.  They are all valid or
            // the tail of the tensor cuts the group, in which case bytes are stored singly.
            bool group_full = ((base + u * 256) | 15u) < total_chunks;
            if (pack_scales && group_full) {
                if ((lane & 15) == 0) *(uint32_t *)(s + soff[u]) = packed;
            } else if ((lane & 3) == 0) {
                s[soff[u]] = (uint8_t)byte;
            }
        }
    }
}

// (T, H, D) attention operand, blocks along D: the row quantizer with a head stride and an
// optional per-(head, channel) fp32 mean subtracted in registers (the smoothing of the MXFP8
// QK^T operands: no shifted copy of the operand reaches memory).  Outputs are contiguous
// (T, H*D) codes and (T, H*D/32) scale bytes.  D % 32 == 0, so a chunk of 8 stays inside a head.
template <int DT, bool SMOOTH>
__global__ __launch_bounds__(256) void quant_heads_kernel(const void *__restrict__ x, uint32_t chunks_per_row,
                                                           uint32_t chunks_per_head, int64_t stride_t, int64_t stride_h,
                                                           const float *__restrict__ mu, uint8_t *__restrict__ q,
                                                           uint8_t *__restrict__ s, uint32_t total_chunks,
                                                           int pack_scales) {
    typedef typename Elem<DT>::type T;
    constexpr int U = 4;
    const int lane = threadIdx.x & 63;
    const uint32_t base = blockIdx.x * (uint32_t)(U * 256) + threadIdx.x;
    float v[U][8];
    bool ok[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const uint32_t chunk = base + u * 256;
        ok[u] = chunk < total_chunks;
        const uint32_t row = chunk / chunks_per_row, col = chunk - row * chunks_per_row;
        const uint32_t head = col / chunks_per_head, d = col - head * chunks_per_head;
        if (ok[u]) {
            Elem<DT>::load8((const T *)x + (int64_t)row * stride_t + (int64_t)head * stride_h + (int64_t)d * 8, v[u]);
            if (SMOOTH) {
                const v4f a = ((const v4f *)(mu + (int64_t)col * 8))[0], b = ((const v4f *)(mu + (int64_t)col * 8))[1];
#pragma unroll
                for (int i = 0; i < 4; i++) v[u][i] -= a[i], v[u][4 + i] -= b[i];
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++) v[u][i] = 0.0f;
        }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
        const uint32_t chunk = base + u * 256;
        float amax = quad_max(amax8(v[u]));
        uint32_t byte = scale_byte(amax);
        const float scale = block_scale(byte);
        uint32_t packed = gather_row_scales(byte, lane);
        if (ok[u]) {
            v2i codes;
            codes[0] = (int)pack4_e4m3(v[u][0], v[u][1], v[u][2], v[u][3], scale);
            codes[1] = (int)pack4_e4m3(v[u][4], v[u][5], v[u][6], v[u][7], scale);
            *(v2i *)(q + (int64_t)chunk * 8) = codes;
            bool group_full = (chunk | 15u) < total_chunks;
            if (pack_scales && group_full) {
                if ((lane & 15) == 0) *(uint32_t *)(s + (chunk >> 2)) = packed;
            } else if ((lane & 3) == 0) {
                s[chunk >> 2] = (uint8_t)byte;
            }
        }
    }
}

// Any strides: one thread per block.  The slow path for doubly-strided views.
template <int DT>
__global__ __launch_bounds__(256) void quant_rows_generic_kernel(const void *__restrict__ x, int64_t M, int64_t KB,
                                                                  int64_t sx_row, int64_t sx_col,
                                                                  uint8_t *__restrict__ q, int64_t ldq,
                                                                  uint8_t *__restrict__ s, int64_t lds) {
    typedef typename Elem<DT>::type T;
    int64_t blk = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (blk >= M * KB) return;
    int64_t row = blk / KB, kb = blk - row * KB;
    const T *p = (const T *)x + row * sx_row + kb * MX_BLOCK * sx_col;
    float v[MX_BLOCK];
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < MX_BLOCK; i++) {
        v[i] = Elem<DT>::load1(p + i * sx_col);
        amax = fmaxf(amax, fabsf(v[i]));
    }
    uint32_t byte = scale_byte(amax);
    const float scale = block_scale(byte);
    uint8_t *qo = q + row * ldq + kb * MX_BLOCK;
#pragma unroll
    for (int i = 0; i < MX_BLOCK; i += 4) {
        uint32_t c = pack4_e4m3(v[i], v[i + 1], v[i + 2], v[i + 3], scale);
        qo[i] = (uint8_t)c;
        qo[i + 1] = (uint8_t)(c >> 8);
        qo[i + 2] = (uint8_t)(c >> 16);
        qo[i + 3] = (uint8_t)(c >> 24);
    }
    s[row * lds + kb] = (uint8_t)byte;
}

// ------------------------------------------------------------------------------------
// Column axis (and dual).  A 256-thread workgroup owns a 128 (M) x 128 (K) tile.  Thread
// (cg = t%16, rg = t/16) holds rows rg*8..+7 x columns cg*8..+7, so wave w holds exactly
// the w-th 32-row block of the tile: the column amax is an in-register max over 8 rows
// and a max across the wave's 4 row groups (lanes l, l^16, l^32, l^48).  Codes are
// transposed through LDS so the (K,M) output is written in full 128-byte rows.
//
// The same with R = 4 rows per thread: a 128 (M) x 64 (K) tile, thread (cg = t%8, rg = t/8)
// holds rows rg*4..+3 x columns cg*8..+7, wave w again the w-th 32-row block (8 row groups:
// lanes l^8, l^16, l^32).  Half the values per thread, half the registers (63 against 90 for
// both axes, 98 against 162 for SwiGLU'), twice the resident waves -- and slower: inside a
// feed-forward step on 16384 x 1536 / 16384 x 4096 bf16, both axes 28.5 against 26.8 us, SwiGLU
// 91.8 against 80.8, SwiGLU' 172.9 against 149.3.  A tile row of 64 columns is a 128-byte run
// where R = 8 reads and writes 256-byte ones, and every scale row is cut into twice as many
// pieces.  Bit-identical results; R = 8 is what the launchers below instantiate.
// ------------------------------------------------------------------------------------

#define QC_TILE 128
#define QC_PITCH 136  // bytes per transposed LDS row (8-byte aligned, staggers banks)

struct QuantTileOut {
    uint8_t *qT;  // (K,M) codes, blocks along M
    int64_t ldqT;
    uint8_t *sT;  // (K,M/32)
    int64_t ldsT;
    uint8_t *q;  // (M,K) codes, blocks along K (only when ROWS)
    int64_t ldq;
    uint8_t *s;  // (M,K/32)
    int64_t lds;
    int pack_row_scales, pack_col_scales;
    // Stage-major code layouts (0: row-major with the pitches above).  q_ks: 128-column panels
    // of q, panel p at p * q_ks, row m of it at m * 128.  qT_ks: the same for qT (panels of 128
    // of its M columns).  A GEMM then finds a K stage of a tile in one contiguous run.
    int64_t q_ks, qT_ks;
};

// Quantizes the 128 x TK tile (TK = 16 R columns) held as v[R][8] per thread (rows m0 + rg*R + i,
// columns kc0 + cg*8 + c of the OUTPUT matrix, which has K columns and M rows) along the column
// axis, and along the row axis too when ROWS.  The token axis is MT long, M rounded up by the
// caller to whole blocks or more: the tile holds zeros for rows past M, they are quantized along
// the columns like any other, and have no row-axis output.  `tile`/`tscale` are the workgroup's LDS
// staging buffers; the caller must not touch them until the function's trailing barrier.
// EDGE = false: no matrix of the launch ends inside a tile (M, MT and K are multiples of the tile), and the stores carry no
// tests.  us with the tests / without, bf16: both axes of 16384 x 4096 55.4 / 54.6, of 8192 x 2048 15.1 / 14.6, of 4096 x 512
// 6.9 / 6.4; SwiGLU 4096 x 4096 22.1 / 21.2.
// COLS: the columns are tested (see the SwiGLU' kernel for the one that keeps the test without EDGE).
template <int R>
struct TileGeom {
    static_assert(R == 8 || R == 4, "8 rows x 8 columns or 4 rows x 8 columns per thread");
    static constexpr int CGS = 2 * R;        // column groups (of 8) across the tile: lanes of one tile row
    static constexpr int TK = 8 * CGS;       // tile columns
    static constexpr int RGS = 256 / CGS;    // row groups (of R rows): 128 rows
    static __device__ __forceinline__ int cg(int t) { return t % CGS; }
    static __device__ __forceinline__ int rg(int t) { return t / CGS; }
};

template <bool ROWS, int R, bool NTS, bool EDGE, bool COLS = EDGE>  // NTS: the code stores carry the non-temporal hint
__device__ __forceinline__ void quant_tile(float (&v)[R][8], const QuantTileOut &o, int64_t M, int64_t MT, int64_t K, int64_t m0,
                                           int64_t kc0, uint8_t *tile, uint8_t *tscale) {
    typedef TileGeom<R> G;
    const int t = threadIdx.x;
    const int lane = t & 63, wave = t >> 6;
    const int cg = G::cg(t), rg = G::rg(t);
    const int64_t col = kc0 + cg * 8;
    const int64_t row0 = m0 + rg * R;
    const bool col_ok = !COLS || col < K;
    const bool whole = !EDGE || m0 + QC_TILE <= M;  // uniform: every row of the tile exists

    if (ROWS) {
        // Row-axis outputs: the 4 lanes of a quad hold 32 consecutive columns of a row.
#pragma unroll
        for (int i = 0; i < R; i++) {
            float amax = quad_max(amax8(v[i]));
            uint32_t byte = scale_byte(amax);
            const float scale = block_scale(byte);
            // the scale bytes of a tile row in one word: four (R = 8, 16 lanes) or two (R = 4, 8 lanes)
            uint32_t packed;
            if (R == 8) {
                packed = gather_row_scales(byte, lane);
            } else {
                packed = byte << ((lane & 4) << 1);
                // row_ror:12 = every lane takes the word of the lane 4 above it in its 16-lane row: lane 0 (8) of a tile
                // row gets block 1's byte from lane 4 (12)
                packed |= (uint32_t)__builtin_amdgcn_mov_dpp((int)packed, 0x12C, 0xF, 0xF, true);
            }
            if (col_ok && (whole || row0 + i < M)) {
                v2i codes;
                codes[0] = (int)pack4_e4m3(v[i][0], v[i][1], v[i][2], v[i][3], scale);
                codes[1] = (int)pack4_e4m3(v[i][4], v[i][5], v[i][6], v[i][7], scale);
                stream_store<NTS>((v2i *)(o.q + (o.q_ks ? (col >> 7) * o.q_ks + (row0 + i) * 128 + (col & 127) : (row0 + i) * o.ldq + col)), codes);
                uint8_t *sp = o.s + (row0 + i) * o.lds + (col >> 5);
                bool full = !EDGE || kc0 + G::TK <= K;
                if (o.pack_row_scales && full) {
                    if (cg == 0) {
                        if (R == 8) *(uint32_t *)sp = packed;
                        else *(uint16_t *)sp = (uint16_t)packed;
                    }
                } else if ((cg & 3) == 0) {
                    *sp = (uint8_t)byte;
                }
            }
        }
    }

    // Column amax over this wave's 32 rows.
    float cm[8];
#pragma unroll
    for (int c = 0; c < 8; c++) {
        float a = fmaxf(fabsf(v[0][c]), fabsf(v[1][c]));
#pragma unroll
        for (int i = 2; i < R; i++) a = fmaxf(a, fabsf(v[i][c]));
        cm[c] = a;
    }
#pragma unroll
    for (int c = 0; c < 8; c++) {
        if (R == 4) {  // lane ^ 8: the other half of the 16-lane row
            const int x = __builtin_amdgcn_mov_dpp((int)f2bits(cm[c]), 0x128, 0xF, 0xF, true);  // row_ror:8
            cm[c] = fmaxf(cm[c], bits2f((uint32_t)x));
        }
        cm[c] = fmaxf(cm[c], __shfl_xor(cm[c], 16, 64));
        cm[c] = fmaxf(cm[c], __shfl_xor(cm[c], 32, 64));
    }
#pragma unroll
    for (int c = 0; c < 8; c++) {
        uint32_t byte = scale_byte(cm[c]);
        const float scale = block_scale(byte);
        uint8_t *dst = tile + (cg * 8 + c) * QC_PITCH + rg * R;
        if (R == 8) {
            v2i codes;
            codes[0] = (int)pack4_e4m3(v[0][c], v[1][c], v[2][c], v[3][c], scale);
            codes[1] = (int)pack4_e4m3(v[R - 4][c], v[R - 3][c], v[R - 2][c], v[R - 1][c], scale);
            *(v2i *)dst = codes;
        } else {
            *(uint32_t *)dst = pack4_e4m3(v[0][c], v[1][c], v[2][c], v[3][c], scale);
        }
        if (rg % (32 / R) == 0) tscale[(cg * 8 + c) * 4 + wave] = (uint8_t)byte;
    }
    __syncthreads();

    // Transposed codes: TK rows of 128 bytes, 16 bytes per thread per pass.
#pragma unroll
    for (int j = 0; j < G::TK / 32; j++) {
        int kr = j * 32 + (t >> 3), ch = t & 7;
        if (!EDGE || (kc0 + kr < K && m0 + ch * 16 < MT)) {
            const v2i *src = (const v2i *)(tile + kr * QC_PITCH + ch * 16);
            v4i w;
            v2i a = src[0], b = src[1];
            w[0] = a[0];
            w[1] = a[1];
            w[2] = b[0];
            w[3] = b[1];
            stream_store<NTS>((v4i *)(o.qT + (o.qT_ks ? (m0 >> 7) * o.qT_ks + (kc0 + kr) * 128 : (kc0 + kr) * o.ldqT + m0) + ch * 16), w);
        }
    }
    if (t < G::TK && (!EDGE || kc0 + t < K)) {
        uint8_t *sp = o.sT + (kc0 + t) * o.ldsT + (m0 >> 5);
        int64_t nb = EDGE ? (MT - m0) >> 5 : 4;
        if (o.pack_col_scales && nb >= 4) {
            *(uint32_t *)sp = *(const uint32_t *)(tscale + t * 4);
        } else {
            for (int b = 0; b < 4 && b < nb; b++) sp[b] = tscale[t * 4 + b];
        }
    }
    __syncthreads();
}

// quant_tile<ROWS, 8, NTS, EDGE> for a tile of 16-bit values kept as loaded (r[i]: row i's eight values, packed): every value
// is converted where it is used, three times instead of once, and the thread holds 32 registers of tile instead of 64.
// The plain row + token axis quantizer then fits 64 registers and eight waves per SIMD (90 registers and five with the
// tile in fp32), so that the 1536 tiles of a 16384 x 1536 activation are resident at once instead of in 1.2 rounds.
// Same arithmetic on the same values: bit-identical outputs.  gate (token axis alone): a factor for each of the thread's rows.
// COLS: the columns are tested in front of the row stores (see quant_cols_kernel for who keeps the test without EDGE).
template <int DT, bool ROWS, bool NTS, bool EDGE, bool COLS = EDGE>
__device__ __forceinline__ void quant_tile_raw(typename Elem<DT>::raw (&r)[8], const QuantTileOut &o, int64_t M, int64_t MT,
                                               int64_t K, int64_t m0, int64_t kc0, uint8_t *tile, uint8_t *tscale,
                                               const float *gate = nullptr) {
    typedef TileGeom<8> G;
    typedef Elem<DT> E;
    const int t = threadIdx.x;
    const int lane = t & 63, wave = t >> 6;
    const int cg = G::cg(t), rg = G::rg(t);
    const int64_t col = kc0 + cg * 8;
    const int64_t row0 = m0 + rg * 8;
    const bool col_ok = !COLS || col < K, whole = !EDGE || m0 + QC_TILE <= M;

    if (ROWS) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            float v[8];
#pragma unroll
            for (int c = 0; c < 8; c++) v[c] = E::elem(r[i], c);
            const float amax = quad_max(amax8(v));
            const uint32_t byte = scale_byte(amax);
            const float scale = block_scale(byte);
            const uint32_t packed = gather_row_scales(byte, lane);
            if (col_ok && (whole || row0 + i < M)) {
                v2i codes;
                codes[0] = (int)pack4_e4m3(v[0], v[1], v[2], v[3], scale);
                codes[1] = (int)pack4_e4m3(v[4], v[5], v[6], v[7], scale);
                stream_store<NTS>((v2i *)(o.q + (o.q_ks ? (col >> 7) * o.q_ks + (row0 + i) * 128 + (col & 127) : (row0 + i) * o.ldq + col)), codes);
                uint8_t *sp = o.s + (row0 + i) * o.lds + (col >> 5);
                const bool full = !EDGE || kc0 + G::TK <= K;
                if (o.pack_row_scales && full) {
                    if (cg == 0) *(uint32_t *)sp = packed;
                } else if ((cg & 3) == 0) {
                    *sp = (uint8_t)byte;
                }
            }
        }
    }
    // The column pass converts the raw values again.  Without this the compiler keeps the 64 conversions of the row
    // pass alive for it, which is the register cost this function exists to avoid.
#pragma unroll
    for (int i = 0; i < 8; i++) asm volatile("" : "+v"(r[i]));
#pragma unroll
    for (int c = 0; c < 8; c++) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = gate ? E::elem(r[i], c) * gate[i] : E::elem(r[i], c);
        float cm = amax8(v);
        cm = fmaxf(cm, __shfl_xor(cm, 16, 64));
        cm = fmaxf(cm, __shfl_xor(cm, 32, 64));
        const uint32_t byte = scale_byte(cm);
        const float scale = block_scale(byte);
        v2i codes;
        codes[0] = (int)pack4_e4m3(v[0], v[1], v[2], v[3], scale);
        codes[1] = (int)pack4_e4m3(v[4], v[5], v[6], v[7], scale);
        *(v2i *)(tile + (cg * 8 + c) * QC_PITCH + rg * 8) = codes;
        if ((rg & 3) == 0) tscale[(cg * 8 + c) * 4 + wave] = (uint8_t)byte;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < G::TK / 32; j++) {
        const int kr = j * 32 + (t >> 3), ch = t & 7;
        if (!EDGE || (kc0 + kr < K && m0 + ch * 16 < MT)) {
            const v2i *src = (const v2i *)(tile + kr * QC_PITCH + ch * 16);
            const v2i a = src[0], b = src[1];
            stream_store<NTS>((v4i *)(o.qT + (o.qT_ks ? (m0 >> 7) * o.qT_ks + (kc0 + kr) * 128 : (kc0 + kr) * o.ldqT + m0) + ch * 16),
                              v4i{a[0], a[1], b[0], b[1]});
        }
    }
    if (t < G::TK && (!EDGE || kc0 + t < K)) {
        uint8_t *sp = o.sT + (kc0 + t) * o.ldsT + (m0 >> 5);
        const int64_t nb = EDGE ? (MT - m0) >> 5 : 4;
        if (o.pack_col_scales && nb >= 4) {
            *(uint32_t *)sp = *(const uint32_t *)(tscale + t * 4);
        } else {
            for (int b = 0; b < 4 && b < nb; b++) sp[b] = tscale[t * 4 + b];
        }
    }
    __syncthreads();
}

// Loads the thread's R rows of 8 values of one operand raw (all loads in flight before any conversion).
template <int DT, int R, bool NT>
__device__ __forceinline__ void load_rows(const void *x, int64_t first, int64_t ld, typename Elem<DT>::raw (&r)[R]) {
    typedef typename Elem<DT>::type T;
#pragma unroll
    for (int i = 0; i < R; i++) r[i] = Elem<DT>::template load_raw<NT>((const T *)x + first + i * ld);
}

// The same for a tile that the matrix may end in: `rows` of the thread's R rows exist (all of them when it is R or more,
// none when it is not positive), the others come back as zeros.  Straight-line code on purpose: rows that do not exist
// read the last one that does (or the matrix's first element) and are zeroed by selects.  With branches around the loads
// the compiler converted the tile in every branch and held it twice (the SwiGLU' kernel: 256 registers instead of 162).
// EDGE = false: a launch whose matrix ends in no tile (rows and columns multiples of 128, nothing padded) needs none of it;
// the selects cost the SwiGLU kernels 2 % of their time there.
template <int DT, int R, bool NT, bool EDGE>
__device__ __forceinline__ void load_rows_or_last(const void *x, int64_t first, int64_t ld, int64_t rows, typename Elem<DT>::raw (&r)[R]) {
    typedef typename Elem<DT>::type T;
    if constexpr (!EDGE) {
        load_rows<DT, R, NT>(x, first, ld, r);
        return;
    }
    const int n = rows < R ? (int)(rows > 0 ? rows : 0) : R;
    const T *const base = (const T *)x + (n ? first : 0);
#pragma unroll
    for (int i = 0; i < R; i++) r[i] = Elem<DT>::template load_raw<NT>(base + (i < n ? i : n ? n - 1 : 0) * ld);
}
template <int DT, int R, bool NT, bool EDGE>
__device__ __forceinline__ void load_rows_or_zero(const void *x, int64_t first, int64_t ld, int64_t rows, typename Elem<DT>::raw (&r)[R]) {
    load_rows_or_last<DT, R, NT, EDGE>(x, first, ld, rows, r);
    if constexpr (!EDGE) return;
#pragma unroll
    for (int i = 0; i < R; i++) {
        typedef int bits_t __attribute__((ext_vector_type(sizeof(r[i]) / 4)));
        const bits_t bits = __builtin_bit_cast(bits_t, r[i]);
        bits_t kept;
#pragma unroll
        for (int e = 0; e < (int)sizeof(r[i]) / 4; e++) kept[e] = i < rows ? bits[e] : 0;
        r[i] = __builtin_bit_cast(typename Elem<DT>::raw, kept);
    }
}

// RAW (16-bit inputs, R = 8): the tile stays packed as loaded (quant_tile_raw): 64 registers, eight waves per SIMD.
// x has M rows and KV columns, the outputs MT and K (both rounded up by the caller): what lies past x is zero.
// CDT: the type fp32 values are rounded to before they are quantized (MX_FP32: none).
// COLS: the thread's loads and row stores stand behind a test of its tile, also where every tile is whole (see launch_cols).
template <int DT, bool DUAL, int R, bool EDGE, bool RAW = false, int CDT = MX_FP32, bool COLS = EDGE>
__global__ __launch_bounds__(256) void quant_cols_kernel(const void *__restrict__ x, int64_t M, int64_t MT, int64_t KV, int64_t K,
                                                          int64_t ldx, QuantTileOut o) {
    typedef TileGeom<R> G;
    __shared__ __attribute__((aligned(16))) uint8_t tile[G::TK * QC_PITCH];
    __shared__ __attribute__((aligned(4))) uint8_t tscale[G::TK * 4];
    const int t = threadIdx.x;
    const int64_t m0 = (int64_t)blockIdx.y * QC_TILE, k0 = (int64_t)blockIdx.x * G::TK;
    const int64_t col = k0 + G::cg(t) * 8;
    const int64_t row0 = m0 + G::rg(t) * R;
    // the thread's loads go out together (row by row, each waited for the one before it)
    typename Elem<DT>::raw r[R];
    // both axes at once is the activation path of a training step, where the 16-bit input is not read again soon: its
    // loads carry the non-temporal hint; the codes are read by the next GEMM and are stored plainly
    if constexpr (COLS && !EDGE) {
        if (col < KV && row0 < M) load_rows<DT, R, DUAL>(x, row0 * ldx + col, ldx, r);  // always so
    } else {
        load_rows_or_zero<DT, R, DUAL, EDGE>(x, row0 * ldx + col, ldx, col < KV ? M - row0 : 0, r);
    }
    if constexpr (RAW) {
        static_assert(DT != MX_FP32 && R == 8, "a packed tile of 16-bit values");
        quant_tile_raw<DT, DUAL, false, EDGE, COLS>(r, o, M, MT, K, m0, k0, tile, tscale);
        return;
    }
    float v[R][8];
#pragma unroll
    for (int i = 0; i < R; i++) {
        Elem<DT>::unpack(r[i], v[i]);
        round_values<CDT>(v[i]);
    }
    quant_tile<DUAL, R, false, EDGE>(v, o, M, MT, K, m0, k0, tile, tscale);
}

// Several matrices of the same rows quantized as the column panels of one (M, K) matrix: what the gradients of projections
// that share an input are to the products of their backward, which contract over (or have rows for) all of them together.
// HBM-bound like quant_cols_kernel, whose tiles these are (every width is a multiple of 128, so a tile has one source);
// 32768 x (2048 + 512 + 512): 77 us in one launch against 53 + 18 + 17 in three.
#define MX_SIDE_MAX 8
struct SideArgs {
    const void *x[MX_SIDE_MAX];
    int64_t ldx[MX_SIDE_MAX];
    int tile_end[MX_SIDE_MAX];  // column tiles of sources 0..j
    int count;
};

template <int DT, bool EDGE, bool RAW, bool COLS = EDGE>  // COLS as in quant_cols_kernel
__global__ __launch_bounds__(256) void quant_side_kernel(SideArgs a, int64_t M, int64_t MT, int64_t K, QuantTileOut o) {
    typedef TileGeom<8> G;
    typedef typename Elem<DT>::type T;
    __shared__ __attribute__((aligned(16))) uint8_t tile[G::TK * QC_PITCH];
    __shared__ __attribute__((aligned(4))) uint8_t tscale[G::TK * 4];
    const int t = threadIdx.x;
    int j = 0;
    while (j + 1 < a.count && (int)blockIdx.x >= a.tile_end[j]) j++;
    const int64_t m0 = (int64_t)blockIdx.y * QC_TILE, k0 = (int64_t)blockIdx.x * G::TK;
    const int64_t col = k0 - (int64_t)(j ? a.tile_end[j - 1] : 0) * G::TK + G::cg(t) * 8;
    const int64_t row0 = m0 + G::rg(t) * 8;
    typename Elem<DT>::raw r[8];
    if constexpr (COLS && !EDGE) {
        if (row0 < M) load_rows<DT, 8, true>(a.x[j], row0 * a.ldx[j] + col, a.ldx[j], r);  // always so
    } else {
        load_rows_or_zero<DT, 8, true, EDGE>(a.x[j], row0 * a.ldx[j] + col, a.ldx[j], M - row0, r);
    }
    if constexpr (RAW) {
        quant_tile_raw<DT, true, false, EDGE, COLS>(r, o, M, MT, K, m0, k0, tile, tscale);
        return;
    }
    float v[8][8];
#pragma unroll
    for (int i = 0; i < 8; i++) Elem<DT>::unpack(r[i], v[i]);
    quant_tile<true, 8, false, EDGE>(v, o, M, MT, K, m0, k0, tile, tscale);
}

// Column panels of one code matrix (codes (rows, K), scale bytes (rows, K/32)) copied together from several: 16 codes per
// thread, every eighth one the four scale bytes of 128 codes too.  Latency-bound at the sizes of weights: 2048 x (2048 + 512 +
// 512) 6.9 us.
struct JoinArgs {
    const uint8_t *codes[MX_SIDE_MAX], *scales[MX_SIDE_MAX];
    int64_t ld[MX_SIDE_MAX], lds[MX_SIDE_MAX];
    int chunk_end[MX_SIDE_MAX];  // 16-code chunks of a row of sources 0..j
    int count;
};

__global__ __launch_bounds__(256) void join_codes_kernel(JoinArgs a, uint32_t total, uint32_t chunks_per_row, uint8_t *__restrict__ codes,
                                                          int64_t ld, uint8_t *__restrict__ scales, int64_t lds) {
    const uint32_t id = blockIdx.x * 256u + threadIdx.x;
    if (id >= total) return;
    const uint32_t row = id / chunks_per_row;
    const int chunk = (int)(id - row * chunks_per_row);
    int j = 0;
    while (j + 1 < a.count && chunk >= a.chunk_end[j]) j++;
    const int from = chunk - (j ? a.chunk_end[j - 1] : 0);
    *(v4i *)(codes + (int64_t)row * ld + (int64_t)chunk * 16) = *(const v4i *)(a.codes[j] + (int64_t)row * a.ld[j] + (int64_t)from * 16);
    if (!(chunk & 7))
        *(uint32_t *)(scales + (int64_t)row * lds + chunk / 2) = *(const uint32_t *)(a.scales[j] + (int64_t)row * a.lds[j] + from / 2);
}

// RMSNorm in front of both quantizers: y = (x * rstd[row]) * w[col] in fp32 -- the two products in the order
// rmsnorm_quant_kernel forms them, so the row-axis pair equals that kernel's bit for bit -- then the tile quantizer.
// rstd comes from a first pass over x (mx_rmsnorm_quantize asked for nothing else); the second read of an activation
// that fits the last-level cache is served from there.  Neither the 16-bit normalized activation nor a transposed copy
// of it reaches memory.
template <int DT, int WDT>
__global__ __launch_bounds__(256) void rmsnorm_quant_dual_kernel(const void *__restrict__ x, int64_t M, int64_t K, int64_t ldx,
                                                                  const void *__restrict__ w, const float *__restrict__ rstd,
                                                                  QuantTileOut o) {
    typedef TileGeom<8> G;
    typedef typename Elem<WDT>::type TW;
    __shared__ __attribute__((aligned(16))) uint8_t tile[G::TK * QC_PITCH];
    __shared__ __attribute__((aligned(4))) uint8_t tscale[G::TK * 4];
    const int t = threadIdx.x;
    const int64_t m0 = (int64_t)blockIdx.y * QC_TILE, k0 = (int64_t)blockIdx.x * G::TK;
    const int64_t col = k0 + G::cg(t) * 8;
    const int64_t row0 = m0 + G::rg(t) * 8;
    const bool ok = col < K && m0 + (t >> 6) * 32 < M;  // K % 8 == 0 and M % 32 == 0
    float v[8][8];
    typename Elem<DT>::raw r[8];
    float wv[8], rs[8];
    if (ok) {
        load_rows<DT, 8, false>(x, row0 * ldx + col, ldx, r);
        const v4f r0 = *(const v4f *)(rstd + row0), r1 = *(const v4f *)(rstd + row0 + 4);
#pragma unroll
        for (int i = 0; i < 4; i++) rs[i] = r0[i], rs[4 + i] = r1[i];
        if (w) {
            Elem<WDT>::load8((const TW *)w + col, wv);
        } else {
#pragma unroll
            for (int c = 0; c < 8; c++) wv[c] = 1.0f;
        }
    }
#pragma unroll
    for (int i = 0; i < 8; i++) {
        if (ok) {
            Elem<DT>::unpack(r[i], v[i]);
#pragma unroll
            for (int c = 0; c < 8; c++) v[i][c] = w ? v[i][c] * rs[i] * wv[c] : v[i][c] * rs[i];
        } else {
#pragma unroll
            for (int c = 0; c < 8; c++) v[i][c] = 0.0f;
        }
    }
    quant_tile<true, 8, false, true>(v, o, M, M, K, m0, k0, tile, tscale);
}

// Several matrices behind one launch: workgroup `id` finds its matrix in the running tile
// totals and quantizes one 128 x 128 tile of it along both axes.  For the once-per-step
// requantization of all weight matrices of a model, where a launch per matrix (and per axis)
// costs more than the bytes it moves.
#define MX_QUANT_BATCH_MAX 24
struct QuantBatchArgs {
    const void *x[MX_QUANT_BATCH_MAX];
    int64_t M[MX_QUANT_BATCH_MAX], K[MX_QUANT_BATCH_MAX], ldx[MX_QUANT_BATCH_MAX];
    QuantTileOut o[MX_QUANT_BATCH_MAX];
    int tile_end[MX_QUANT_BATCH_MAX];  // tiles of problems 0..j
    int tiles_k[MX_QUANT_BATCH_MAX];
    int count;
};

template <int DT>
__global__ __launch_bounds__(256) void quant_dual_batch_kernel(QuantBatchArgs b) {
    typedef typename Elem<DT>::type T;
    __shared__ __attribute__((aligned(16))) uint8_t tile[QC_TILE * QC_PITCH];
    __shared__ __attribute__((aligned(4))) uint8_t tscale[QC_TILE * 4];
    const int t = threadIdx.x;
    int j = 0;
    while (j + 1 < b.count && (int)blockIdx.x >= b.tile_end[j]) j++;
    const int local = (int)blockIdx.x - (j ? b.tile_end[j - 1] : 0);
    const int64_t M = b.M[j], K = b.K[j], ldx = b.ldx[j];
    const void *x = b.x[j];
    const int64_t m0 = (int64_t)(local / b.tiles_k[j]) * QC_TILE, k0 = (int64_t)(local % b.tiles_k[j]) * QC_TILE;
    const int64_t col = k0 + (t & 15) * 8;
    const int64_t row0 = m0 + (t >> 4) * 8;
    const bool ok = col < K && m0 + (t >> 6) * 32 < M;
    float v[8][8];
    typename Elem<DT>::raw r[8];  // eight loads in flight, then the conversions
    if (ok) {
#pragma unroll
        for (int i = 0; i < 8; i++) r[i] = Elem<DT>::load_raw((const T *)x + (row0 + i) * ldx + col);
    }
#pragma unroll
    for (int i = 0; i < 8; i++) {
        if (ok) {
            Elem<DT>::unpack(r[i], v[i]);
        } else {
#pragma unroll
            for (int c = 0; c < 8; c++) v[i][c] = 0.0f;
        }
    }
    quant_tile<true, 8, false, true>(v, b.o[j], M, M, K, m0, k0, tile, tscale);
}

__device__ __forceinline__ float sigmoid_fast(float x) { return sigmoid_f32(x); }

// h = silu(g) * u from the fused projection output gu (M, 2H) (gate half first), quantized
// along both axes: (q,s) (M,H) for the down projection's forward, (qT,sT) (H,MT) for its wgrad.
// ROUNDED: silu(g) and the product are rounded to the input type one after the other, as the two
// 16-bit operators of an unfused activation leave them; otherwise h stays in fp32 up to the cast.
template <int DT, int R, bool ROUNDED, bool EDGE>
__global__ __launch_bounds__(256) void swiglu_quant_dual_kernel(const void *__restrict__ gu, int64_t M, int64_t MT, int64_t H,
                                                                 int64_t ldgu, QuantTileOut o) {
    typedef TileGeom<R> G;
    __shared__ __attribute__((aligned(16))) uint8_t tile[G::TK * QC_PITCH];
    __shared__ __attribute__((aligned(4))) uint8_t tscale[G::TK * 4];
    const int t = threadIdx.x;
    const int64_t m0 = (int64_t)blockIdx.y * QC_TILE, k0 = (int64_t)blockIdx.x * G::TK;
    const int64_t col = k0 + G::cg(t) * 8;
    const int64_t row0 = m0 + G::rg(t) * R;
    const int64_t rows = col < H ? M - row0 : 0;
    float v[R][8];
    typename Elem<DT>::raw rg[R], ru[R];  // all loads in flight before the first conversion
    load_rows_or_zero<DT, R, true, EDGE>(gu, row0 * ldgu + col, ldgu, rows, rg);
    load_rows_or_zero<DT, R, true, EDGE>(gu, row0 * ldgu + H + col, ldgu, rows, ru);
#pragma unroll
    for (int i = 0; i < R; i++) {  // zeros give zeros
        float g[8], u[8];
        Elem<DT>::unpack(rg[i], g);
        Elem<DT>::unpack(ru[i], u);
        if constexpr (ROUNDED) {
#pragma unroll
            for (int c = 0; c < 8; c++) v[i][c] = g[c] * sigmoid_fast(g[c]);
            round_values<DT>(v[i]);
#pragma unroll
            for (int c = 0; c < 8; c++) v[i][c] *= u[c];
            round_values<DT>(v[i]);
        } else {
#pragma unroll
            for (int c = 0; c < 8; c++) v[i][c] = g[c] * sigmoid_fast(g[c]) * u[c];
        }
    }
    // hundreds of MB in, hundreds out, nothing of it small enough to be found in a cache by its consumer: all hinted
    quant_tile<true, R, true, EDGE>(v, o, M, MT, H, m0, k0, tile, tscale);
}

// SwiGLU backward fused with both quantizers.  Reads dh (M,H) and the saved projection
// output gu (M,2H); forms dgate = dh * u * s * (1 + g (1 - s)) and dup = dh * g * s with
// s = sigmoid(g) in fp32 (elementwise/swiglu.py:108-119, experts_bwd.py:145-148 of the
// reference); writes dpre = [dgate | dup] quantized along 2H ((q,s): (M,2H)) for the input
// projection's dgrad and along the tokens ((qT,sT): (2H,MT)) for its wgrad.  o.q/o.qT address the
// full (M,2H) / (2H,MT) outputs.  ROUNDED: the gradients of the unfused activation, whose 16-bit
// operators round silu(g), dh * u, dgate and dup to the input type.
template <int DT, int R, bool ROUNDED, bool EDGE>
__global__ __launch_bounds__(256) void swiglu_bwd_quant_dual_kernel(const void *__restrict__ dh, int64_t lddh,
                                                                     const void *__restrict__ gu, int64_t ldgu,
                                                                     int64_t M, int64_t MT, int64_t H, QuantTileOut o) {
    typedef TileGeom<R> G;
    __shared__ __attribute__((aligned(16))) uint8_t tile[G::TK * QC_PITCH];
    __shared__ __attribute__((aligned(4))) uint8_t tscale[G::TK * 4];
    const int t = threadIdx.x;
    const int64_t m0 = (int64_t)blockIdx.y * QC_TILE, k0 = (int64_t)blockIdx.x * G::TK;
    const int64_t col = k0 + G::cg(t) * 8;
    const int64_t row0 = m0 + G::rg(t) * R;
    const int64_t rows = col < H ? M - row0 : 0;
    float v[R][8], w[R][8];
    // All loads of the thread go out before the first conversion.  Written row by row (load three,
    // convert, next row) the compiler kept that order and every thread had 48 bytes in flight at a time,
    // with a memory latency in front of each of its rows.  Rows past the end of the matrix repeat the
    // last one and are left out below.
    typename Elem<DT>::raw rg[R], ru[R], rd[R];
    load_rows_or_last<DT, R, true, EDGE>(gu, row0 * ldgu + col, ldgu, rows, rg);
    load_rows_or_last<DT, R, true, EDGE>(gu, row0 * ldgu + H + col, ldgu, rows, ru);
    load_rows_or_last<DT, R, true, EDGE>(dh, row0 * lddh + col, lddh, rows, rd);
    // waited for here and not row by row, where the stores of the rows before are waited for too (they count alike)
    // (16384 x 4096: 126.1 -> 124.9 us with the tests gone; a matrix that ends in a tile gains nothing: 44.5 and 44.9 us at 5003 x 4096)
    if constexpr (!EDGE) {
#pragma unroll
        for (int i = 0; i < R; i++) asm volatile("" : "+v"(rg[i]), "+v"(ru[i]), "+v"(rd[i]));
    }
#pragma unroll
    for (int i = 0; i < R; i++) {
        if (i < rows) {  // (always so without EDGE: a block per row all the same, or the compiler takes 256 registers for them)
            float g[8], u[8], d[8];
            Elem<DT>::unpack(rg[i], g);
            Elem<DT>::unpack(ru[i], u);
            Elem<DT>::unpack(rd[i], d);
            if constexpr (ROUNDED) {
                float slope[8];
#pragma unroll
                for (int c = 0; c < 8; c++) {
                    const float sg = sigmoid_fast(g[c]);
                    slope[c] = sg * (1.0f + g[c] * (1.0f - sg));
                    w[i][c] = g[c] * sg;
                    v[i][c] = d[c] * u[c];
                }
                round_values<DT>(w[i]);
                round_values<DT>(v[i]);
#pragma unroll
                for (int c = 0; c < 8; c++) {
                    w[i][c] *= d[c];
                    v[i][c] *= slope[c];
                }
                round_values<DT>(w[i]);
                round_values<DT>(v[i]);
            } else {
#pragma unroll
                for (int c = 0; c < 8; c++) {
                    float sg = sigmoid_fast(g[c]);
                    v[i][c] = d[c] * u[c] * sg * (1.0f + g[c] * (1.0f - sg));
                    w[i][c] = d[c] * g[c] * sg;
                }
            }
        } else {
#pragma unroll
            for (int c = 0; c < 8; c++) v[i][c] = w[i][c] = 0.0f;
        }
    }
    // The gate half occupies output columns [0,H), the up half [H,2H): same tile, shifted.
    // Columns at or beyond H inside the gate-half tile are masked by passing K = H.  The column test stays without EDGE: as
    // straight-line code the rows' stores overlap in 175 registers, two waves per SIMD instead of three (16384 x 4096: 134.4 us
    // without it, 124.9 with it).
    quant_tile<true, R, true, EDGE, true>(v, o, M, MT, H, m0, k0, tile, tscale);
    QuantTileOut o2 = o;
    o2.q += o.q_ks ? (H >> 7) * o.q_ks : H;
    o2.s += H / MX_BLOCK;
    o2.qT += o.qT_ks ? H * 128 : H * o.ldqT;
    o2.sT += H * o.ldsT;
    quant_tile<true, R, true, EDGE, true>(w, o2, M, MT, H, m0, k0, tile, tscale);
}

// ------------------------------------------------------------------------------------
// silu(gate) * up in fp32 -> row-axis MXFP8 (fused_act.py:37-66 of the reference).  ROUNDED as in swiglu_quant_dual_kernel.
// ------------------------------------------------------------------------------------

template <int DT, int U, bool ROUNDED>
__global__ __launch_bounds__(256) void swiglu_quant_rows_kernel(const void *__restrict__ g, const void *__restrict__ up,
                                                                 uint32_t chunks_per_row, int64_t ldg, int64_t ldu,
                                                                 uint8_t *__restrict__ q, int64_t ldq,
                                                                 uint8_t *__restrict__ s, int64_t lds,
                                                                 uint32_t total_chunks, int pack_scales) {
    typedef typename Elem<DT>::type T;
    const int lane = threadIdx.x & 63;
    const uint32_t base = blockIdx.x * (uint32_t)(U * 256) + threadIdx.x;
    float a[U][8], b[U][8];
    int64_t qoff[U], soff[U];
    bool ok[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        uint32_t chunk = base + u * 256;
        ok[u] = chunk < total_chunks;
        uint32_t row = chunk / chunks_per_row;
        uint32_t col = chunk - row * chunks_per_row;
        qoff[u] = (int64_t)row * ldq + (int64_t)col * 8;
        soff[u] = (int64_t)row * lds + (col >> 2);
        if (ok[u]) {
            Elem<DT>::load8((const T *)g + (int64_t)row * ldg + (int64_t)col * 8, a[u]);
            Elem<DT>::load8((const T *)up + (int64_t)row * ldu + (int64_t)col * 8, b[u]);
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++) a[u][i] = b[u][i] = 0.0f;
        }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            float gv = a[u][i];
            v[i] = gv * sigmoid_f32(gv);
        }
        if constexpr (ROUNDED) round_values<DT>(v);
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] *= b[u][i];
        if constexpr (ROUNDED) round_values<DT>(v);
        float amax = quad_max(amax8(v));
        uint32_t byte = scale_byte(amax);
        const float scale = block_scale(byte);
        uint32_t packed = gather_row_scales(byte, lane);
        if (ok[u]) {
            v2i codes;
            codes[0] = (int)pack4_e4m3(v[0], v[1], v[2], v[3], scale);
            codes[1] = (int)pack4_e4m3(v[4], v[5], v[6], v[7], scale);
            *(v2i *)(q + qoff[u]) = codes;
            bool group_full = ((base + u * 256) | 15u) < total_chunks;
            if (pack_scales && group_full) {
                if ((lane & 15) == 0) *(uint32_t *)(s + soff[u]) = packed;
            } else if ((lane & 3) == 0) {
                s[soff[u]] = (uint8_t)byte;
            }
        }
    }
}

// ------------------------------------------------------------------------------------
// Column-axis quantizer over expert-sorted rows, for the routed experts' MXFP8 WGRAD.
// WGRAD contracts the rows an expert owns, so the 32-row blocks must not straddle two experts:
// every expert's segment is laid out from a fresh multiple of 128 in a padded position space
// (tile t of 128 rows = positions [128 t, 128 t + 128)), rows past the segment's end are zero.
// Row tile -> (expert, first row) is resolved on the device from `offsets`, like the GEMMs.
// Sources: SRC_PLAIN  x[index[m] or m] (optionally times row_scale[scale_index[m]] in fp32,
//                     the gate applied to dout rows: grouped.py:218-221 of the reference)
//          SRC_SWIGLU silu(pre[m][c]) * pre[m][H + c] in fp32 (moe.py:288-290 rebuilds h from pre)
// ------------------------------------------------------------------------------------

enum { SRC_PLAIN = 0, SRC_SWIGLU = 1 };

struct GroupedQuantArgs {
    const void *x;
    int64_t ldx;
    int C;  // output columns of x to quantize (H for SRC_SWIGLU, whose x has 2H columns)
    const int32_t *index;
    const void *row_scale;
    const int32_t *scale_index;
    int scale_f32;
    const int32_t *offsets;
    int E;
};

// The expert whose tiles contain row tile `rt`: owner[] = expert, its first tile, its first and its end row; owner[0] < 0 for
// a tile past the last one.  The first wave looks at 64 experts at a time (one coalesced read of `offsets`, a wave scan of
// their tile counts) instead of walking the experts with a dependent scalar load each: with hundreds of experts, most of them
// empty, that walk took longer than the tile itself.
__device__ __forceinline__ void tile_owner(const GroupedQuantArgs &a, int rt, int (&owner)[4]) {
    const int t = threadIdx.x;
    if (t < 64) {
        int carry = 0;
        bool done = false;
        for (int e0 = 0; e0 < a.E && !done; e0 += 64) {
            const int e = e0 + t;
            const int lo = e < a.E ? a.offsets[e] : 0, hi = e < a.E ? a.offsets[e + 1] : 0;
            const int tiles = (hi - lo + QC_TILE - 1) / QC_TILE;
            const int incl = wave_incl_scan(tiles, t);
            const int first = carry + incl - tiles;
            const bool mine = e < a.E && rt >= first && rt < first + tiles;
            if (__ballot(mine)) {
                if (mine) owner[0] = e, owner[1] = first, owner[2] = lo, owner[3] = hi;
                done = true;
            }
            carry += __shfl(incl, 63, 64);
        }
        if (!done && t == 0) owner[0] = -1;
    }
    __syncthreads();
}

template <int DT>
__global__ __launch_bounds__(256) void quant_swiglu_grouped_kernel(GroupedQuantArgs a, QuantTileOut o, int64_t mpad) {
    typedef typename Elem<DT>::type T;
    __shared__ __attribute__((aligned(16))) uint8_t tile[QC_TILE * QC_PITCH];
    __shared__ __attribute__((aligned(4))) uint8_t tscale[QC_TILE * 4];
    __shared__ int owner[4];
    const int t = threadIdx.x, rt = blockIdx.y;
    tile_owner(a, rt, owner);
    if (owner[0] < 0) return;  // that part of the padded space is never read
    const int end = owner[3], row_base = owner[2] + (rt - owner[1]) * QC_TILE;
    const int64_t k0 = (int64_t)blockIdx.x * QC_TILE;
    const int64_t col = k0 + (t & 15) * 8;
    const bool col_ok = col < a.C;
    float v[8][8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int pos = row_base + (t >> 4) * 8 + i;
        if (col_ok && pos < end) {
            const int64_t src = a.index ? a.index[pos] : pos;
            float g[8], u[8];
            Elem<DT>::load8((const T *)a.x + src * a.ldx + col, g);
            Elem<DT>::load8((const T *)a.x + src * a.ldx + a.C + col, u);
#pragma unroll
            for (int c = 0; c < 8; c++) v[i][c] = g[c] * sigmoid_fast(g[c]) * u[c];
        } else {
#pragma unroll
            for (int c = 0; c < 8; c++) v[i][c] = 0.0f;
        }
    }
    quant_tile<false, 8, false, true>(v, o, mpad, mpad, a.C, (int64_t)rt * QC_TILE, k0, tile, tscale);
}

// SRC_PLAIN.  Bound by the gathered reads and the code stores; what it lacked was waves in flight.  With the tile in fp32 and
// four column tiles per workgroup it took 166 registers, three waves per SIMD, and the 1664 workgroups of 98304 rows x 1024 ran in
// 2.2 rounds of 768.  Packed as loaded (quant_tile_raw, which converts every value once here), one tile per workgroup, it takes 57
// and eight waves: 98304 rows from 16384 x 1024, us before / now: 96 / 55 with a row scale (GATED), 86 / 53 without; 16662 rows from
// 2777: 25 / 17 and 20 / 15.5.  Four or two tiles per workgroup: 61 and 58, 61 and 55.  (Left to itself the compiler takes 228
// registers for the straight-line form.)
template <int DT, bool GATED>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void quant_cols_grouped_kernel(GroupedQuantArgs a, QuantTileOut o, int64_t mpad) {
    typedef typename Elem<DT>::type T;
    __shared__ __attribute__((aligned(16))) uint8_t tile[QC_TILE * QC_PITCH];
    __shared__ __attribute__((aligned(4))) uint8_t tscale[QC_TILE * 4];
    __shared__ int owner[4];
    const int t = threadIdx.x, rt = blockIdx.y;
    tile_owner(a, rt, owner);
    if (owner[0] < 0) return;  // that part of the padded space is never read
    const int end = owner[3], row_base = owner[2] + (rt - owner[1]) * QC_TILE;
    // each source row's index and scale factor is read by one thread, not by the 16 that hold the row
    __shared__ __attribute__((aligned(16))) int src_of[QC_TILE];
    __shared__ __attribute__((aligned(16))) float gate_of[QC_TILE];
    if (t < QC_TILE) {
        const int pos = row_base + t;
        const bool real = pos < end;
        src_of[t] = !real ? -1 : a.index ? a.index[pos] : pos;
        if constexpr (GATED) {
            const int si = !real ? 0 : a.scale_index ? a.scale_index[pos] : pos;
            gate_of[t] = !real ? 1.0f : a.scale_f32 ? ((const float *)a.row_scale)[si] : Elem<DT>::load1((const T *)a.row_scale + si);
        }
    }
    __syncthreads();
    const int64_t k0 = (int64_t)blockIdx.x * QC_TILE, col = k0 + (t & 15) * 8;
    typename Elem<DT>::raw r[8];
    float gate[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int src = src_of[(t >> 4) * 8 + i];
        gate[i] = GATED ? gate_of[(t >> 4) * 8 + i] : 1.0f;
        r[i] = __builtin_bit_cast(typename Elem<DT>::raw, v4i{0, 0, 0, 0});
        if (col < a.C && src >= 0) r[i] = Elem<DT>::load_raw((const T *)a.x + (int64_t)src * a.ldx + col);
    }
    quant_tile_raw<DT, false, false, true>(r, o, mpad, mpad, a.C, (int64_t)rt * QC_TILE, k0, tile, tscale, GATED ? gate : nullptr);
}

}  // namespace mx

// ------------------------------------------------------------------------------------
// C ABI
// ------------------------------------------------------------------------------------

using namespace mx;

static inline bool aligned(const void *p, uintptr_t a) { return ((uintptr_t)p & (a - 1)) == 0; }
static inline int esize(int dt) { return dt == MX_FP32 ? 4 : 2; }

#define MX_LAUNCH_CHECK()                                   \
    do {                                                    \
        if (hipGetLastError() != hipSuccess) return MX_ELAUNCH; \
    } while (0)

template <int DT, int CDT = MX_FP32>
static int launch_rows(const void *x, int64_t M, int64_t K, int64_t sx_row, int64_t sx_col, uint8_t *q, int64_t ldq,
                       uint8_t *s, int64_t lds, hipStream_t st) {
    const int64_t KB = K / MX_BLOCK;
    const bool vec_ok = sx_col == 1 && aligned(x, 16) && (sx_row * esize(DT)) % 16 == 0 && aligned(q, 8) &&
                        ldq % 8 == 0 && M * (K / 8) < (int64_t)0x7FFFFF00;
    if (!vec_ok) {
        if (CDT != MX_FP32) return MX_EUNSUPPORTED;
        int64_t blocks = M * KB;
        if ((blocks + 255) / 256 > 0x7FFFFFFF) return MX_EUNSUPPORTED;
        quant_rows_generic_kernel<DT><<<dim3((unsigned)((blocks + 255) / 256)), dim3(256), 0, st>>>(
            x, M, KB, sx_row, sx_col, q, ldq, s, lds);
        MX_LAUNCH_CHECK();
        return MX_OK;
    }
    // 16-byte chunks per thread.  Measured on 128 MB and more of bf16: 4 chunks 5.6 TB/s, 2 chunks 6.0, 1 chunk 5.75
    constexpr int U = 2;
    const uint32_t cpr = (uint32_t)(K / 8);
    const uint32_t total = (uint32_t)(M * (K / 8));
    const unsigned grid = (total + U * 256 - 1) / (U * 256);
    const bool flat = sx_row == K && ldq == K && lds == KB;
    if (flat) {
        int pack = aligned(s, 4);
        quant_rows_kernel<DT, U, true, CDT><<<dim3(grid), dim3(256), 0, st>>>(x, cpr, sx_row, q, ldq, s, lds, total, pack);
    } else {
        int pack = aligned(s, 4) && lds % 4 == 0 && KB % 4 == 0;
        quant_rows_kernel<DT, U, false, CDT><<<dim3(grid), dim3(256), 0, st>>>(x, cpr, sx_row, q, ldq, s, lds, total, pack);
    }
    MX_LAUNCH_CHECK();
    return MX_OK;
}

// A leading dimension of exactly 128 for a matrix wider than 128 columns asks for the stage-major
// layout: 128-column panels, each holding every row (pitch 128), panel p at p * rows * 128.
static bool stage_major(int64_t ld, int64_t cols) { return ld == 128 && cols > 128; }

static QuantTileOut tile_out(uint8_t *qT, int64_t ldqT, uint8_t *sT, int64_t ldsT, uint8_t *q, int64_t ldq, uint8_t *s,
                             int64_t lds, int64_t q_ks = 0, int64_t qT_ks = 0) {
    QuantTileOut o;
    o.qT = qT, o.ldqT = ldqT, o.sT = sT, o.ldsT = ldsT, o.q = q, o.ldq = ldq, o.s = s, o.lds = lds;
    o.q_ks = q_ks, o.qT_ks = qT_ks;
    o.pack_row_scales = s != nullptr && aligned(s, 4) && lds % 4 == 0;
    o.pack_col_scales = aligned(sT, 4) && ldsT % 4 == 0;
    return o;
}

// Rows per thread of the dense tile quantizers (see TileGeom): 8 = 128 x 128 tiles.
constexpr int MX_QR_COLS = 8, MX_QR_SWIGLU = 8, MX_QR_SWIGLU_BWD = 8;

template <int R>
static bool tile_grid(int64_t M, int64_t K, dim3 &grid) {
    grid = dim3((unsigned)((K + TileGeom<R>::TK - 1) / TileGeom<R>::TK), (unsigned)((M + QC_TILE - 1) / QC_TILE));
    return grid.y <= 65535u;
}

// x has M rows and KV columns; the outputs span MT (token axis) and K.  cast: the 16-bit type fp32 values are rounded to
// first, MX_FP32 for none.
template <int DT, bool DUAL>
static int launch_cols(const void *x, int64_t M, int64_t MT, int64_t KV, int64_t K, int64_t ldx, uint8_t *qT, int64_t ldqT,
                       uint8_t *sT, int64_t ldsT, uint8_t *q, int64_t ldq, uint8_t *s, int64_t lds, hipStream_t st,
                       int64_t qT_ks = 0, int cast = MX_FP32) {
    dim3 grid;
    if (!tile_grid<MX_QR_COLS>(MT, K, grid)) return MX_EUNSUPPORTED;
    const QuantTileOut o = tile_out(qT, ldqT, sT, ldsT, q, ldq, s, lds, 0, qT_ks);
    // Both axes of a 16-bit matrix whose tiles are all resident at once with eight waves per SIMD, but not with the five
    // the fp32 tile allows, go to the packed-tile kernel: 16384 x 1536 (1536 tiles on 256 CUs) 27.0 -> 24.9 us.  Larger
    // matrices run several rounds either way and are faster with fewer, fatter waves (16384 x 4096: 54.4 against 58.9 us).
    // Launches of whole tiles carry no tests, but for those of more than four and up to six tiles per CU, which are faster
    // with a test around a thread's loads and row stores.  us without / with, bf16: 8192 x 2048 (1024 tiles) 15.1 / 16.0,
    // 9216 x 2048 19.5 / 17.6, 4096 x 5120 (1280) 20.5 / 17.6, 16384 x 1536 24.0 / 23.1, 14336 x 2048 (1792) 26.2 / 26.6,
    // 16384 x 2048 29.3 / 30.6.
    const dim3 block(256);
    const bool edge = M % QC_TILE || K % QC_TILE || MT != M || KV != K;
#define MX_LAUNCH_COLS(...)                                                                                                   \
    (edge ? quant_cols_kernel<DT, DUAL, MX_QR_COLS, true, __VA_ARGS__><<<grid, block, 0, st>>>(x, M, MT, KV, K, ldx, o)       \
          : quant_cols_kernel<DT, DUAL, MX_QR_COLS, false, __VA_ARGS__><<<grid, block, 0, st>>>(x, M, MT, KV, K, ldx, o))
    if constexpr (DT != MX_FP32 && DUAL) {
        const int64_t tiles = (int64_t)grid.x * grid.y, cus = num_cus();
        if (tiles > 4 * cus && tiles <= 6 * cus && !edge)
            quant_cols_kernel<DT, true, MX_QR_COLS, false, true, MX_FP32, true><<<grid, block, 0, st>>>(x, M, MT, KV, K, ldx, o);
        else if (tiles <= 8 * cus) MX_LAUNCH_COLS(true);
        else MX_LAUNCH_COLS(false);
    } else if constexpr (DUAL) {
        if (cast == MX_BF16) MX_LAUNCH_COLS(false, MX_BF16);
        else if (cast == MX_FP16) MX_LAUNCH_COLS(false, MX_FP16);
        else MX_LAUNCH_COLS(false);
    } else {
        MX_LAUNCH_COLS(false);
    }
#undef MX_LAUNCH_COLS
    MX_LAUNCH_CHECK();
    return MX_OK;
}

static bool cols_vec_ok(const void *x, int dt, int64_t K, int64_t ldx, const uint8_t *qT, int64_t ldqT) {
    return K % 8 == 0 && aligned(x, 16) && (ldx * esize(dt)) % 16 == 0 && aligned(qT, 16) && ldqT % 16 == 0;
}

template <int DT>
static int launch_norm_dual(const void *x, int64_t M, int64_t K, int64_t ldx, const void *w, int w_dtype, const float *rstd,
                            const QuantTileOut &o, hipStream_t st) {
    dim3 grid;
    if (!tile_grid<8>(M, K, grid)) return MX_EUNSUPPORTED;
    switch (w ? w_dtype : (int)MX_FP32) {
    case MX_BF16: rmsnorm_quant_dual_kernel<DT, MX_BF16><<<grid, dim3(256), 0, st>>>(x, M, K, ldx, w, rstd, o); break;
    case MX_FP16: rmsnorm_quant_dual_kernel<DT, MX_FP16><<<grid, dim3(256), 0, st>>>(x, M, K, ldx, w, rstd, o); break;
    default: rmsnorm_quant_dual_kernel<DT, MX_FP32><<<grid, dim3(256), 0, st>>>(x, M, K, ldx, w, rstd, o); break;
    }
    MX_LAUNCH_CHECK();
    return MX_OK;
}

extern "C" int mx_rmsnorm_quantize_dual(const void *x, int x_dtype, int64_t M, int64_t K, int64_t ldx, const void *weight,
                                        int w_dtype, float eps, float *rstd, uint8_t *q, int64_t ldq, uint8_t *s,
                                        int64_t lds, uint8_t *qT, int64_t ldqT, uint8_t *sT, int64_t ldsT, void *stream) {
    const bool panels = stage_major(ldqT, M);
    if (M < 0 || K <= 0 || M % MX_BLOCK || K % MX_BLOCK || !x || !rstd || !q || !s || !qT || !sT || ldx < K || ldq < K ||
        lds < K / MX_BLOCK || (ldqT < M && !panels) || (panels && M % 128) || ldsT < M / MX_BLOCK)
        return MX_EINVAL;
    if (x_dtype != MX_BF16 && x_dtype != MX_FP16 && x_dtype != MX_FP32) return MX_EINVAL;
    if (weight && w_dtype != MX_BF16 && w_dtype != MX_FP16 && w_dtype != MX_FP32) return MX_EINVAL;
    if (M == 0) return MX_OK;
    if (!cols_vec_ok(x, x_dtype, K, ldx, qT, ldqT) || !aligned(q, 8) || ldq % 8 || !aligned(rstd, 16) ||
        (weight && !aligned(weight, 16)))
        return MX_EUNSUPPORTED;
    // first pass: the rows' reciprocal root mean squares (the row kernel, asked for nothing but rstd)
    int rc = mx_rmsnorm_quantize(x, x_dtype, M, K, ldx, nullptr, 0, eps, nullptr, 0, rstd, nullptr, 0, nullptr, 0, stream);
    if (rc != MX_OK) return rc;
    hipStream_t st = (hipStream_t)stream;
    const QuantTileOut o = tile_out(qT, ldqT, sT, ldsT, q, ldq, s, lds, 0, panels ? K * 128 : 0);
    switch (x_dtype) {
    case MX_BF16: return launch_norm_dual<MX_BF16>(x, M, K, ldx, weight, w_dtype, rstd, o, st);
    case MX_FP16: return launch_norm_dual<MX_FP16>(x, M, K, ldx, weight, w_dtype, rstd, o, st);
    default: return launch_norm_dual<MX_FP32>(x, M, K, ldx, weight, w_dtype, rstd, o, st);
    }
}

extern "C" int mx_quantize_cols(const void *x, int x_dtype, int64_t M, int64_t K, int64_t ldx, uint8_t *qT,
                                int64_t ldqT, uint8_t *sT, int64_t ldsT, void *stream) {
    if (M < 0 || K < 0 || M % MX_BLOCK || ldx < K || ldqT < M || ldsT < M / MX_BLOCK) return MX_EINVAL;
    if (M == 0 || K == 0) return MX_OK;
    hipStream_t st = (hipStream_t)stream;
    if (mx::stream_is_capturing(st)) return MX_ECAPTURE;
    if (!cols_vec_ok(x, x_dtype, K, ldx, qT, ldqT)) {
        // Rows of the transposed view, one thread per block.
        switch (x_dtype) {
        case MX_BF16: return launch_rows<MX_BF16>(x, K, M, 1, ldx, qT, ldqT, sT, ldsT, st);
        case MX_FP16: return launch_rows<MX_FP16>(x, K, M, 1, ldx, qT, ldqT, sT, ldsT, st);
        case MX_FP32: return launch_rows<MX_FP32>(x, K, M, 1, ldx, qT, ldqT, sT, ldsT, st);
        default: return MX_EINVAL;
        }
    }
    switch (x_dtype) {
    case MX_BF16: return launch_cols<MX_BF16, false>(x, M, M, K, K, ldx, qT, ldqT, sT, ldsT, nullptr, 0, nullptr, 0, st);
    case MX_FP16: return launch_cols<MX_FP16, false>(x, M, M, K, K, ldx, qT, ldqT, sT, ldsT, nullptr, 0, nullptr, 0, st);
    case MX_FP32: return launch_cols<MX_FP32, false>(x, M, M, K, K, ldx, qT, ldqT, sT, ldsT, nullptr, 0, nullptr, 0, st);
    default: return MX_EINVAL;
    }
}

extern "C" int mx_quantize_rows(const void *x, int x_dtype, int64_t M, int64_t K, int64_t sx_row, int64_t sx_col,
                                uint8_t *q, int64_t ldq, uint8_t *s, int64_t lds, void *stream) {
    if (M < 0 || K < 0 || K % MX_BLOCK || ldq < K || lds < K / MX_BLOCK) return MX_EINVAL;
    if (M == 0 || K == 0) return MX_OK;
    hipStream_t st = (hipStream_t)stream;
    if (mx::stream_is_capturing(st)) return MX_ECAPTURE;
    // A transposed view (unit stride down the rows) is the column quantizer of the
    // matrix underneath it: no copy is made.
    if (sx_col != 1 && sx_row == 1 && M > 1 && cols_vec_ok(x, x_dtype, M, sx_col, q, ldq))
        return mx_quantize_cols(x, x_dtype, K, M, sx_col, q, ldq, s, lds, stream);
    switch (x_dtype) {
    case MX_BF16: return launch_rows<MX_BF16>(x, M, K, sx_row, sx_col, q, ldq, s, lds, st);
    case MX_FP16: return launch_rows<MX_FP16>(x, M, K, sx_row, sx_col, q, ldq, s, lds, st);
    case MX_FP32: return launch_rows<MX_FP32>(x, M, K, sx_row, sx_col, q, ldq, s, lds, st);
    default: return MX_EINVAL;
    }
}

template <int DT>
static int launch_heads(const void *x, int64_t T, int64_t H, int64_t D, int64_t stride_t, int64_t stride_h,
                        const float *mu, uint8_t *q, uint8_t *s, hipStream_t st) {
    const uint32_t cpr = (uint32_t)(H * D / 8), cph = (uint32_t)(D / 8), total = (uint32_t)(T * (H * D / 8));
    const unsigned grid = (total + 4 * 256 - 1) / (4 * 256);
    // the outputs are contiguous, so a 16-lane group's 4 scale bytes are one aligned dword whatever the row length
    const int pack = aligned(s, 4);
    if (mu)
        quant_heads_kernel<DT, true><<<dim3(grid), dim3(256), 0, st>>>(x, cpr, cph, stride_t, stride_h, mu, q, s, total, pack);
    else
        quant_heads_kernel<DT, false><<<dim3(grid), dim3(256), 0, st>>>(x, cpr, cph, stride_t, stride_h, mu, q, s, total, pack);
    MX_LAUNCH_CHECK();
    return MX_OK;
}

extern "C" int mx_quantize_heads(const void *x, int x_dtype, int64_t T, int64_t H, int64_t D, int64_t stride_t,
                                 int64_t stride_h, const float *mu, uint8_t *q, uint8_t *s, void *stream) {
    if (T < 0 || H < 0 || D < 0 || D % MX_BLOCK || (H > 1 && stride_h < D) || stride_t < 0) return MX_EINVAL;
    if (x_dtype != MX_BF16 && x_dtype != MX_FP16 && x_dtype != MX_FP32) return MX_EINVAL;
    if (T == 0 || H == 0 || D == 0) return MX_OK;
    if (!x || !q || !s) return MX_EINVAL;
    if (!aligned(x, 16) || (stride_t * esize(x_dtype)) % 16 || (stride_h * esize(x_dtype)) % 16 || !aligned(q, 8) ||
        (mu && !aligned(mu, 16)) || T * (H * D / 8) >= (int64_t)0x7FFFFF00)
        return MX_EUNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    if (mx::stream_is_capturing(st)) return MX_ECAPTURE;
    switch (x_dtype) {
    case MX_BF16: return launch_heads<MX_BF16>(x, T, H, D, stride_t, stride_h, mu, q, s, st);
    case MX_FP16: return launch_heads<MX_FP16>(x, T, H, D, stride_t, stride_h, mu, q, s, st);
    default: return launch_heads<MX_FP32>(x, T, H, D, stride_t, stride_h, mu, q, s, st);
    }
}

extern "C" int mx_quantize_dual(const void *x, int x_dtype, int64_t M, int64_t K, int64_t ldx, uint8_t *q, int64_t ldq,
                                uint8_t *s, int64_t lds, uint8_t *qT, int64_t ldqT, uint8_t *sT, int64_t ldsT,
                                void *stream) {
    const bool panels = stage_major(ldqT, M);  // qT as 128-token panels
    if (M < 0 || K < 0 || M % MX_BLOCK || K % MX_BLOCK || ldx < K || ldq < K || lds < K / MX_BLOCK ||
        (ldqT < M && !panels) || (panels && M % 128) || ldsT < M / MX_BLOCK)
        return MX_EINVAL;
    if (M == 0 || K == 0) return MX_OK;
    hipStream_t st = (hipStream_t)stream;
    if (mx::stream_is_capturing(st)) return MX_ECAPTURE;
    if (!cols_vec_ok(x, x_dtype, K, ldx, qT, ldqT) || !aligned(q, 8) || ldq % 8) {
        if (panels) return MX_EUNSUPPORTED;
        int rc = mx_quantize_rows(x, x_dtype, M, K, ldx, 1, q, ldq, s, lds, stream);
        if (rc != MX_OK) return rc;
        return mx_quantize_cols(x, x_dtype, M, K, ldx, qT, ldqT, sT, ldsT, stream);
    }
    const int64_t ks = panels ? K * 128 : 0;
    switch (x_dtype) {
    case MX_BF16: return launch_cols<MX_BF16, true>(x, M, M, K, K, ldx, qT, ldqT, sT, ldsT, q, ldq, s, lds, st, ks);
    case MX_FP16: return launch_cols<MX_FP16, true>(x, M, M, K, K, ldx, qT, ldqT, sT, ldsT, q, ldq, s, lds, st, ks);
    case MX_FP32: return launch_cols<MX_FP32, true>(x, M, M, K, K, ldx, qT, ldqT, sT, ldsT, q, ldq, s, lds, st, ks);
    default: return MX_EINVAL;
    }
}

extern "C" int mx_quantize_dual_batch(const mx_quant_problem *problems, int count, int x_dtype, void *stream) {
    if (count < 0 || (count > 0 && !problems)) return MX_EINVAL;
    if (x_dtype != MX_BF16 && x_dtype != MX_FP16 && x_dtype != MX_FP32) return MX_EINVAL;
    for (int j = 0; j < count; j++) {  // validate everything before launching anything
        const mx_quant_problem &p = problems[j];
        if (p.M < 0 || p.K < 0 || p.M % MX_BLOCK || p.K % MX_BLOCK || p.ldx < p.K || p.ldq < p.K ||
            p.lds < p.K / MX_BLOCK || p.ldqT < p.M || p.ldsT < p.M / MX_BLOCK)
            return MX_EINVAL;
        if (p.M && p.K && (!p.x || !p.q || !p.s || !p.qT || !p.sT)) return MX_EINVAL;
    }
    hipStream_t st = (hipStream_t)stream;
    if (mx::stream_is_capturing(st)) return MX_ECAPTURE;
    QuantBatchArgs b;
    b.count = 0;
    int64_t total = 0;
    auto flush = [&]() -> int {
        if (b.count) {
            const dim3 grid((unsigned)total), block(256);
            switch (x_dtype) {
            case MX_BF16: quant_dual_batch_kernel<MX_BF16><<<grid, block, 0, st>>>(b); break;
            case MX_FP16: quant_dual_batch_kernel<MX_FP16><<<grid, block, 0, st>>>(b); break;
            default: quant_dual_batch_kernel<MX_FP32><<<grid, block, 0, st>>>(b); break;
            }
            MX_LAUNCH_CHECK();
        }
        b.count = 0, total = 0;
        return MX_OK;
    };
    for (int j = 0; j < count; j++) {
        const mx_quant_problem &p = problems[j];
        if (p.M == 0 || p.K == 0) continue;
        const int64_t tiles_k = (p.K + QC_TILE - 1) / QC_TILE, tiles = tiles_k * ((p.M + QC_TILE - 1) / QC_TILE);
        if (!cols_vec_ok(p.x, x_dtype, p.K, p.ldx, p.qT, p.ldqT) || !aligned(p.q, 8) || p.ldq % 8 ||
            tiles > 0x3FFFFFFF) {
            // an operand the tiled kernel does not take goes through the single-matrix entry point
            int rc = mx_quantize_dual(p.x, x_dtype, p.M, p.K, p.ldx, p.q, p.ldq, p.s, p.lds, p.qT, p.ldqT, p.sT, p.ldsT,
                                      stream);
            if (rc != MX_OK) return rc;
            continue;
        }
        if (b.count == MX_QUANT_BATCH_MAX || total + tiles > 0x3FFFFFFF) {
            int rc = flush();
            if (rc != MX_OK) return rc;
        }
        const int k = b.count++;
        b.x[k] = p.x, b.M[k] = p.M, b.K[k] = p.K, b.ldx[k] = p.ldx;
        b.o[k] = tile_out(p.qT, p.ldqT, p.sT, p.ldsT, p.q, p.ldq, p.s, p.lds);
        total += tiles;
        b.tile_end[k] = (int)total, b.tiles_k[k] = (int)tiles_k;
    }
    return flush();
}

template <int DT, bool ROUNDED>
static int launch_swiglu(const void *g, const void *u, int64_t M, int64_t K, int64_t ldg, int64_t ldu, uint8_t *q,
                         int64_t ldq, uint8_t *s, int64_t lds, hipStream_t st) {
    constexpr int U = 2;
    const uint32_t total = (uint32_t)(M * (K / 8));
    const unsigned grid = (total + U * 256 - 1) / (U * 256);
    int pack = aligned(s, 4) && lds % 4 == 0 && (K / MX_BLOCK) % 4 == 0;
    swiglu_quant_rows_kernel<DT, U, ROUNDED><<<dim3(grid), dim3(256), 0, st>>>(g, u, (uint32_t)(K / 8), ldg, ldu, q, ldq, s, lds,
                                                                      total, pack);
    MX_LAUNCH_CHECK();
    return MX_OK;
}

extern "C" int mx_swiglu_quantize_rows(const void *gate, const void *up, int dtype, int64_t M, int64_t K, int64_t ldg,
                                       int64_t ldu, uint8_t *q, int64_t ldq, uint8_t *s, int64_t lds, void *stream) {
    if (M < 0 || K < 0 || K % MX_BLOCK || ldg < K || ldu < K || ldq < K || lds < K / MX_BLOCK) return MX_EINVAL;
    if (M == 0 || K == 0) return MX_OK;
    if (dtype != MX_BF16 && dtype != MX_FP16) return MX_EUNSUPPORTED;
    if (!aligned(gate, 16) || !aligned(up, 16) || (ldg * 2) % 16 || (ldu * 2) % 16 || !aligned(q, 8) || ldq % 8 ||
        M * (K / 8) >= (int64_t)0x7FFFFF00)
        return MX_EUNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    if (mx::stream_is_capturing(st)) return MX_ECAPTURE;
    return dtype == MX_BF16 ? launch_swiglu<MX_BF16, false>(gate, up, M, K, ldg, ldu, q, ldq, s, lds, st)
                            : launch_swiglu<MX_FP16, false>(gate, up, M, K, ldg, ldu, q, ldq, s, lds, st);
}

template <int DT, bool ROUNDED>
static int launch_swiglu_dual(const void *gu, int64_t M, int64_t MT, int64_t H, int64_t ldgu, dim3 grid, const QuantTileOut &o, hipStream_t st) {
    constexpr int R = MX_QR_SWIGLU;
    if (M % QC_TILE || H % QC_TILE || MT != M) swiglu_quant_dual_kernel<DT, R, ROUNDED, true><<<grid, dim3(256), 0, st>>>(gu, M, MT, H, ldgu, o);
    else swiglu_quant_dual_kernel<DT, R, ROUNDED, false><<<grid, dim3(256), 0, st>>>(gu, M, MT, H, ldgu, o);
    MX_LAUNCH_CHECK();
    return MX_OK;
}

static int launch_swiglu_dual(const void *gu, int dtype, int64_t M, int64_t MT, int64_t H, int64_t ldgu, int rounded, dim3 grid,
                              const QuantTileOut &o, hipStream_t st) {
    if (dtype == MX_BF16)
        return rounded ? launch_swiglu_dual<MX_BF16, true>(gu, M, MT, H, ldgu, grid, o, st) : launch_swiglu_dual<MX_BF16, false>(gu, M, MT, H, ldgu, grid, o, st);
    return rounded ? launch_swiglu_dual<MX_FP16, true>(gu, M, MT, H, ldgu, grid, o, st) : launch_swiglu_dual<MX_FP16, false>(gu, M, MT, H, ldgu, grid, o, st);
}

template <int DT, bool ROUNDED>
static int launch_swiglu_bwd_dual(const void *dh, int64_t lddh, const void *gu, int64_t ldgu, int64_t M, int64_t MT, int64_t H, dim3 grid,
                                  const QuantTileOut &o, hipStream_t st) {
    constexpr int R = MX_QR_SWIGLU_BWD;
    if (M % QC_TILE || H % QC_TILE || MT != M)
        swiglu_bwd_quant_dual_kernel<DT, R, ROUNDED, true><<<grid, dim3(256), 0, st>>>(dh, lddh, gu, ldgu, M, MT, H, o);
    else swiglu_bwd_quant_dual_kernel<DT, R, ROUNDED, false><<<grid, dim3(256), 0, st>>>(dh, lddh, gu, ldgu, M, MT, H, o);
    MX_LAUNCH_CHECK();
    return MX_OK;
}

static int launch_swiglu_bwd_dual(const void *dh, int64_t lddh, const void *gu, int64_t ldgu, int dtype, int64_t M, int64_t MT,
                                  int64_t H, int rounded, dim3 grid, const QuantTileOut &o, hipStream_t st) {
    if (dtype == MX_BF16)
        return rounded ? launch_swiglu_bwd_dual<MX_BF16, true>(dh, lddh, gu, ldgu, M, MT, H, grid, o, st)
                       : launch_swiglu_bwd_dual<MX_BF16, false>(dh, lddh, gu, ldgu, M, MT, H, grid, o, st);
    return rounded ? launch_swiglu_bwd_dual<MX_FP16, true>(dh, lddh, gu, ldgu, M, MT, H, grid, o, st)
                   : launch_swiglu_bwd_dual<MX_FP16, false>(dh, lddh, gu, ldgu, M, MT, H, grid, o, st);
}

extern "C" int mx_swiglu_quantize_dual(const void *gu, int dtype, int64_t M, int64_t H, int64_t ldgu, uint8_t *q,
                                       int64_t ldq, uint8_t *s, int64_t lds, uint8_t *qT, int64_t ldqT, uint8_t *sT,
                                       int64_t ldsT, void *stream) {
    const bool panels = stage_major(ldqT, M);  // qT as 128-token panels
    if (M < 0 || H < 0 || M % MX_BLOCK || H % MX_BLOCK || ldgu < 2 * H || ldq < H || lds < H / MX_BLOCK ||
        (ldqT < M && !panels) || (panels && M % 128) || ldsT < M / MX_BLOCK)
        return MX_EINVAL;
    if (M == 0 || H == 0) return MX_OK;
    if (dtype != MX_BF16 && dtype != MX_FP16) return MX_EUNSUPPORTED;
    if (!aligned(gu, 16) || (ldgu * 2) % 16 || !aligned(q, 8) || ldq % 8 || !aligned(qT, 16) || ldqT % 16)
        return MX_EUNSUPPORTED;
    dim3 grid;
    if (!tile_grid<MX_QR_SWIGLU>(M, H, grid)) return MX_EUNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    if (mx::stream_is_capturing(st)) return MX_ECAPTURE;
    QuantTileOut o = tile_out(qT, ldqT, sT, ldsT, q, ldq, s, lds, 0, panels ? H * 128 : 0);
    return launch_swiglu_dual(gu, dtype, M, M, H, ldgu, 0, grid, o, st);
}

extern "C" int mx_swiglu_bwd_quantize_dual(const void *dh, int64_t lddh, const void *gu, int64_t ldgu, int dtype,
                                           int64_t M, int64_t H, uint8_t *q, int64_t ldq, uint8_t *s, int64_t lds,
                                           uint8_t *qT, int64_t ldqT, uint8_t *sT, int64_t ldsT, void *stream) {
    const bool q_panels = stage_major(ldq, 2 * H), qt_panels = stage_major(ldqT, M);
    if (M < 0 || H < 0 || M % MX_BLOCK || H % MX_BLOCK || lddh < H || ldgu < 2 * H || (ldq < 2 * H && !q_panels) ||
        (q_panels && H % 128) || lds < 2 * H / MX_BLOCK || (ldqT < M && !qt_panels) || (qt_panels && M % 128) ||
        ldsT < M / MX_BLOCK)
        return MX_EINVAL;
    if (M == 0 || H == 0) return MX_OK;
    if (dtype != MX_BF16 && dtype != MX_FP16) return MX_EUNSUPPORTED;
    if (!aligned(gu, 16) || (ldgu * 2) % 16 || !aligned(dh, 16) || (lddh * 2) % 16 || !aligned(q, 8) || ldq % 8 ||
        !aligned(qT, 16) || ldqT % 16)
        return MX_EUNSUPPORTED;
    dim3 grid;
    if (!tile_grid<MX_QR_SWIGLU_BWD>(M, H, grid)) return MX_EUNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    if (mx::stream_is_capturing(st)) return MX_ECAPTURE;
    QuantTileOut o = tile_out(qT, ldqT, sT, ldsT, q, ldq, s, lds, q_panels ? M * 128 : 0, qt_panels ? 2 * H * 128 : 0);
    if (H % 128) o.pack_row_scales = 0;  // the up half's scale columns start at H/32: keep the packed stores aligned
    return launch_swiglu_bwd_dual(dh, lddh, gu, ldgu, dtype, M, M, H, 0, grid, o, st);
}

// ------------------------------------------------------------------------------------
// The activation quantizers of a training step: any row count, token-axis operand in whole 128-token panels.  Without a
// token-axis operand (qT and sT null: a forward nobody will differentiate, or frozen weights) they are the row kernels:
// half the bytes and no transposition.  us both axes / rows: 8 x 2048 6.4 / 2.4, 1500 x 1536 8.4 / 3.6, SwiGLU of 1500 x 4096
// 11.6 / 6.5.
// ------------------------------------------------------------------------------------

static bool token_extent_ok(int64_t M, int64_t MT) { return M > 0 && MT >= M && MT % QC_TILE == 0; }

extern "C" int mx_quantize_tokens(const void *x, int x_dtype, int cast_dtype, int64_t M, int64_t KV, int64_t ldx, int64_t MT,
                                  int64_t K, uint8_t *q, int64_t ldq, uint8_t *s, int64_t lds, uint8_t *qT, uint8_t *sT,
                                  int64_t ldsT, void *stream) {
    const bool rows_only = !qT && !sT;
    if (!token_extent_ok(M, MT) || KV <= 0 || KV > K || K % MX_BLOCK || !x || !q || !s || (!rows_only && (!qT || !sT)) || ldx < KV ||
        ldq < K || lds < K / MX_BLOCK || (!rows_only && ldsT < MT / MX_BLOCK) || (cast_dtype != x_dtype && x_dtype != MX_FP32))
        return MX_EINVAL;
    if (rows_only) {
        if (KV != K || M * (K / 8) >= (int64_t)0x7FFFFF00) return MX_EUNSUPPORTED;
        hipStream_t st = (hipStream_t)stream;
        if (mx::stream_is_capturing(st)) return MX_ECAPTURE;
        switch (x_dtype) {
        case MX_BF16: return launch_rows<MX_BF16>(x, M, K, ldx, 1, q, ldq, s, lds, st);
        case MX_FP16: return launch_rows<MX_FP16>(x, M, K, ldx, 1, q, ldq, s, lds, st);
        case MX_FP32:
            return cast_dtype == MX_BF16   ? launch_rows<MX_FP32, MX_BF16>(x, M, K, ldx, 1, q, ldq, s, lds, st)
                   : cast_dtype == MX_FP16 ? launch_rows<MX_FP32, MX_FP16>(x, M, K, ldx, 1, q, ldq, s, lds, st)
                                           : launch_rows<MX_FP32>(x, M, K, ldx, 1, q, ldq, s, lds, st);
        default: return MX_EINVAL;
        }
    }
    if (KV % 8 || !cols_vec_ok(x, x_dtype, K, ldx, qT, 128) || !aligned(q, 8) || ldq % 8) return MX_EUNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    if (mx::stream_is_capturing(st)) return MX_ECAPTURE;
    const int64_t ks = K * 128;
    switch (x_dtype) {
    case MX_BF16: return launch_cols<MX_BF16, true>(x, M, MT, KV, K, ldx, qT, 128, sT, ldsT, q, ldq, s, lds, st, ks);
    case MX_FP16: return launch_cols<MX_FP16, true>(x, M, MT, KV, K, ldx, qT, 128, sT, ldsT, q, ldq, s, lds, st, ks);
    case MX_FP32: return launch_cols<MX_FP32, true>(x, M, MT, KV, K, ldx, qT, 128, sT, ldsT, q, ldq, s, lds, st, ks, cast_dtype);
    default: return MX_EINVAL;
    }
}

template <int DT>
static int launch_side(const SideArgs &a, int64_t M, int64_t MT, int64_t K, dim3 grid, const QuantTileOut &o, hipStream_t st) {
    const int64_t tiles = (int64_t)grid.x * grid.y, cus = num_cus();
    // as launch_cols; without / with the tests, K = 3072: 6144 rows (1152 tiles) 20.1 / 17.9 us, 8192 24.2 / 23.3, 9216 26.3 / 27.5
    const bool raw = tiles <= 8 * cus, tested = tiles > 4 * cus && tiles <= 6 * cus;
    const dim3 block(256);
    if (M != MT) {
        if (raw) quant_side_kernel<DT, true, true><<<grid, block, 0, st>>>(a, M, MT, K, o);
        else quant_side_kernel<DT, true, false><<<grid, block, 0, st>>>(a, M, MT, K, o);
    } else {
        if (raw && tested) quant_side_kernel<DT, false, true, true><<<grid, block, 0, st>>>(a, M, MT, K, o);
        else if (raw) quant_side_kernel<DT, false, true><<<grid, block, 0, st>>>(a, M, MT, K, o);
        else quant_side_kernel<DT, false, false><<<grid, block, 0, st>>>(a, M, MT, K, o);
    }
    MX_LAUNCH_CHECK();
    return MX_OK;
}

extern "C" int mx_quantize_tokens_side(const mx_side_source *sources, int count, int x_dtype, int64_t M, int64_t MT, uint8_t *q,
                                       int64_t ldq, uint8_t *s, int64_t lds, uint8_t *qT, uint8_t *sT, int64_t ldsT, void *stream) {
    if (count < 1 || count > MX_SIDE_MAX || !sources || !token_extent_ok(M, MT) || !q || !s || !qT || !sT || ldsT < MT / MX_BLOCK ||
        (x_dtype != MX_BF16 && x_dtype != MX_FP16))
        return MX_EINVAL;
    SideArgs a;
    int64_t tiles = 0;
    bool vec = aligned(q, 16) && ldq % 16 == 0 && aligned(qT, 16);
    for (int j = 0; j < count; j++) {
        const mx_side_source &p = sources[j];
        if (!p.x || p.K <= 0 || p.K % QC_TILE || p.ldx < p.K) return MX_EINVAL;
        tiles += p.K / QC_TILE;
        if (tiles > 0x7FFFFF) return MX_EUNSUPPORTED;
        vec = vec && aligned(p.x, 16) && p.ldx % 8 == 0;
        a.x[j] = p.x, a.ldx[j] = p.ldx, a.tile_end[j] = (int)tiles;
    }
    a.count = count;
    const int64_t K = tiles * QC_TILE;
    if (ldq < K || lds < K / MX_BLOCK) return MX_EINVAL;
    dim3 grid;
    if (!vec || !tile_grid<8>(MT, K, grid)) return MX_EUNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    if (mx::stream_is_capturing(st)) return MX_ECAPTURE;
    const QuantTileOut o = tile_out(qT, 128, sT, ldsT, q, ldq, s, lds, 0, K * 128);
    return x_dtype == MX_BF16 ? launch_side<MX_BF16>(a, M, MT, K, grid, o, st) : launch_side<MX_FP16>(a, M, MT, K, grid, o, st);
}

extern "C" int mx_join_codes(const mx_code_source *sources, int count, int64_t rows, uint8_t *codes, int64_t ld, uint8_t *scales,
                             int64_t lds, void *stream) {
    if (count < 1 || count > MX_SIDE_MAX || !sources || rows <= 0 || !codes || !scales) return MX_EINVAL;
    JoinArgs a;
    int64_t chunks = 0;
    bool vec = aligned(codes, 16) && ld % 16 == 0 && aligned(scales, 4) && lds % 4 == 0;
    for (int j = 0; j < count; j++) {
        const mx_code_source &p = sources[j];
        if (!p.codes || !p.scales || p.K <= 0 || p.K % 128 || p.ld < p.K || p.lds < p.K / MX_BLOCK) return MX_EINVAL;
        chunks += p.K / 16;
        if (chunks * rows >= (int64_t)0x7FFFFF00) return MX_EUNSUPPORTED;
        vec = vec && aligned(p.codes, 16) && p.ld % 16 == 0 && aligned(p.scales, 4) && p.lds % 4 == 0;
        a.codes[j] = p.codes, a.scales[j] = p.scales, a.ld[j] = p.ld, a.lds[j] = p.lds, a.chunk_end[j] = (int)chunks;
    }
    a.count = count;
    if (ld < chunks * 16 || lds < chunks / 2) return MX_EINVAL;
    if (!vec) return MX_EUNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    if (mx::stream_is_capturing(st)) return MX_ECAPTURE;
    const uint32_t total = (uint32_t)(chunks * rows);
    join_codes_kernel<<<dim3((total + 255) / 256), dim3(256), 0, st>>>(a, total, (uint32_t)chunks, codes, ld, scales, lds);
    MX_LAUNCH_CHECK();
    return MX_OK;
}

extern "C" int mx_swiglu_quantize_tokens(const void *gu, int dtype, int rounded, int64_t M, int64_t H, int64_t ldgu, int64_t MT,
                                         uint8_t *q, int64_t ldq, uint8_t *s, int64_t lds, uint8_t *qT, uint8_t *sT,
                                         int64_t ldsT, void *stream) {
    const bool rows_only = !qT && !sT;
    if (!token_extent_ok(M, MT) || H <= 0 || H % MX_BLOCK || !gu || !q || !s || (!rows_only && (!qT || !sT)) || ldgu < 2 * H ||
        ldq < H || lds < H / MX_BLOCK || (!rows_only && ldsT < MT / MX_BLOCK))
        return MX_EINVAL;
    if (rows_only) {
        const uint8_t *const up = (const uint8_t *)gu + H * 2;
        if ((dtype != MX_BF16 && dtype != MX_FP16) || !aligned(gu, 16) || (ldgu * 2) % 16 || !aligned(q, 8) || ldq % 8 ||
            M * (H / 8) >= (int64_t)0x7FFFFF00)
            return MX_EUNSUPPORTED;
        hipStream_t st = (hipStream_t)stream;
        if (mx::stream_is_capturing(st)) return MX_ECAPTURE;
        if (dtype == MX_BF16)
            return rounded ? launch_swiglu<MX_BF16, true>(gu, up, M, H, ldgu, ldgu, q, ldq, s, lds, st)
                           : launch_swiglu<MX_BF16, false>(gu, up, M, H, ldgu, ldgu, q, ldq, s, lds, st);
        return rounded ? launch_swiglu<MX_FP16, true>(gu, up, M, H, ldgu, ldgu, q, ldq, s, lds, st)
                       : launch_swiglu<MX_FP16, false>(gu, up, M, H, ldgu, ldgu, q, ldq, s, lds, st);
    }
    if ((dtype != MX_BF16 && dtype != MX_FP16) || !aligned(gu, 16) || (ldgu * 2) % 16 || !aligned(q, 8) || ldq % 8 || !aligned(qT, 16))
        return MX_EUNSUPPORTED;
    dim3 grid;
    if (!tile_grid<MX_QR_SWIGLU>(MT, H, grid)) return MX_EUNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    if (mx::stream_is_capturing(st)) return MX_ECAPTURE;
    return launch_swiglu_dual(gu, dtype, M, MT, H, ldgu, rounded, grid, tile_out(qT, 128, sT, ldsT, q, ldq, s, lds, 0, H * 128), st);
}

extern "C" int mx_swiglu_bwd_quantize_tokens(const void *dh, int64_t lddh, const void *gu, int64_t ldgu, int dtype, int rounded,
                                             int64_t M, int64_t H, int64_t MT, uint8_t *q, int64_t ldq, uint8_t *s, int64_t lds,
                                             uint8_t *qT, uint8_t *sT, int64_t ldsT, void *stream) {
    const bool q_panels = stage_major(ldq, 2 * H);
    if (!token_extent_ok(M, MT) || H <= 0 || H % MX_BLOCK || !dh || !gu || !q || !s || !qT || !sT || lddh < H || ldgu < 2 * H ||
        (ldq < 2 * H && !q_panels) || (q_panels && H % 128) || lds < 2 * H / MX_BLOCK || ldsT < MT / MX_BLOCK)
        return MX_EINVAL;
    if ((dtype != MX_BF16 && dtype != MX_FP16) || !aligned(gu, 16) || (ldgu * 2) % 16 || !aligned(dh, 16) || (lddh * 2) % 16 ||
        !aligned(q, 8) || ldq % 8 || !aligned(qT, 16))
        return MX_EUNSUPPORTED;
    dim3 grid;
    if (!tile_grid<MX_QR_SWIGLU_BWD>(MT, H, grid)) return MX_EUNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    if (mx::stream_is_capturing(st)) return MX_ECAPTURE;
    QuantTileOut o = tile_out(qT, 128, sT, ldsT, q, ldq, s, lds, q_panels ? M * 128 : 0, 2 * H * 128);
    if (H % 128) o.pack_row_scales = 0;  // the up half's scale columns start at H/32: keep the packed stores aligned
    return launch_swiglu_bwd_dual(dh, lddh, gu, ldgu, dtype, M, MT, H, rounded, grid, o, st);
}

extern "C" int mx_quantize_cols_grouped(const void *x, int dtype, int64_t ldx, int64_t C, int source,
                                        const int32_t *index, const void *row_scale, int row_scale_dtype,
                                        const int32_t *scale_index, const int32_t *offsets, int64_t E, int64_t M,
                                        uint8_t *qT, int64_t ldqT, uint8_t *sT, int64_t ldsT, void *stream) {
    if (M < 0 || C < 0 || E <= 0 || E >= (1 << 20) || M >= 0x7FFFFFFF || C >= 0x7FFFFFFF) return MX_EINVAL;
    if (source != SRC_PLAIN && source != SRC_SWIGLU) return MX_EINVAL;
    const int64_t tiles = (M + QC_TILE - 1) / QC_TILE + E;
    const int64_t mpad = tiles * QC_TILE;
    // a leading dimension of exactly 128 on the wider padded axis: qT stage-major, (Mpad/128, C, 128)
    const bool qt_panels = ldqT == 128 && mpad > 128;
    if ((ldqT < mpad && !qt_panels) || ldsT < mpad / MX_BLOCK || ldx < (source == SRC_SWIGLU ? 2 * C : C)) return MX_EINVAL;
    if (row_scale && row_scale_dtype != MX_FP32 && row_scale_dtype != dtype) return MX_EINVAL;
    if (dtype != MX_BF16 && dtype != MX_FP16) return MX_EUNSUPPORTED;
    if (C % 8 || !aligned(x, 16) || (ldx * 2) % 16 || !aligned(qT, 16) || ldqT % 16 || tiles > 65535) return MX_EUNSUPPORTED;
    if (C == 0) return MX_OK;
    GroupedQuantArgs a;
    a.x = x, a.ldx = ldx, a.C = (int)C, a.index = index, a.row_scale = row_scale, a.scale_index = scale_index;
    a.scale_f32 = row_scale_dtype == MX_FP32, a.offsets = offsets, a.E = (int)E;
    QuantTileOut o = tile_out(qT, ldqT, sT, ldsT, nullptr, 0, nullptr, 0, 0, qt_panels ? C * 128 : 0);
    const int ctiles = (int)((C + QC_TILE - 1) / QC_TILE);
    const dim3 grid((unsigned)ctiles, (unsigned)tiles);
    hipStream_t st = (hipStream_t)stream;
    if (mx::stream_is_capturing(st)) return MX_ECAPTURE;
#define MX_QCG_LAUNCH(DT)                                                                                                      \
    (source == SRC_SWIGLU ? quant_swiglu_grouped_kernel<DT><<<grid, dim3(256), 0, st>>>(a, o, mpad)                            \
     : row_scale          ? quant_cols_grouped_kernel<DT, true><<<grid, dim3(256), 0, st>>>(a, o, mpad)                        \
                          : quant_cols_grouped_kernel<DT, false><<<grid, dim3(256), 0, st>>>(a, o, mpad))
    if (dtype == MX_BF16) MX_QCG_LAUNCH(MX_BF16);
    else MX_QCG_LAUNCH(MX_FP16);
#undef MX_QCG_LAUNCH
    MX_LAUNCH_CHECK();
    return MX_OK;
}

// ---- cuBLAS SWIZZLE_32_4_4 scale layout (interop) -------------------------------------------------
// 128-row x 4-column tiles of 512 bytes, row-tile major; inside a tile scale (r, c) sits at
// (r % 32) * 16 + (r / 32) * 4 + c; zero padded to whole tiles.  One thread moves the 4 bytes
// of one row of one tile.  (src/kohakuwullm/kernels/mxfp8/interop.py:24-41, quantize.py:175-180.)
namespace mx {
template <bool TO_SWIZZLED>
__global__ __launch_bounds__(256) void swizzle_scales_kernel(uint8_t *__restrict__ natural, int64_t lds,
                                                             uint8_t *__restrict__ swizzled, int64_t rows, int64_t cols,
                                                             int64_t col_tiles, int64_t total) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;  // one dword of the swizzled buffer
    if (idx >= total) return;
    const int64_t tile = idx >> 7;
    const int in = (int)(idx & 127);        // (r % 32) * 4 + r / 32
    const int rr = (in >> 2) + 32 * (in & 3);
    const int64_t r = (tile / col_tiles) * 128 + rr;
    const int64_t c0 = (tile % col_tiles) * 4;
    if (TO_SWIZZLED) {
        uint32_t w = 0;
        if (r < rows)
            for (int c = 0; c < 4; c++)
                if (c0 + c < cols) w |= (uint32_t)natural[r * lds + c0 + c] << (8 * c);
        ((uint32_t *)swizzled)[idx] = w;
    } else if (r < rows) {
        const uint32_t w = ((const uint32_t *)swizzled)[idx];
        for (int c = 0; c < 4; c++)
            if (c0 + c < cols) natural[r * lds + c0 + c] = (uint8_t)(w >> (8 * c));
    }
}
}  // namespace mx

static int swizzle_launch(bool to_swizzled, uint8_t *natural, int64_t lds, uint8_t *swizzled, int64_t rows, int64_t cols,
                          void *stream) {
    if (rows < 0 || cols < 0 || lds < cols) return MX_EINVAL;
    if (((uintptr_t)swizzled & 3) != 0) return MX_EINVAL;
    const int64_t row_tiles = (rows + 127) / 128, col_tiles = (cols + 3) / 4;
    const int64_t total = row_tiles * col_tiles * 128;
    if (total == 0) return MX_OK;
    const int64_t blocks = (total + 255) / 256;
    if (blocks > 0x7FFFFFFF) return MX_EUNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    if (mx::stream_is_capturing(st)) return MX_ECAPTURE;
    if (to_swizzled)
        mx::swizzle_scales_kernel<true><<<dim3((unsigned)blocks), dim3(256), 0, st>>>(natural, lds, swizzled, rows, cols,
                                                                                    col_tiles, total);
    else
        mx::swizzle_scales_kernel<false><<<dim3((unsigned)blocks), dim3(256), 0, st>>>(natural, lds, swizzled, rows, cols,
                                                                                     col_tiles, total);
    return hipGetLastError() == hipSuccess ? MX_OK : MX_ELAUNCH;
}

extern "C" int mx_swizzle_scales(const uint8_t *s, int64_t rows, int64_t cols, int64_t lds, uint8_t *swizzled,
                                 void *stream) {
    return swizzle_launch(true, (uint8_t *)s, lds, swizzled, rows, cols, stream);
}

extern "C" int mx_unswizzle_scales(const uint8_t *swizzled, int64_t rows, int64_t cols, uint8_t *s, int64_t lds,
                                   void *stream) {
    return swizzle_launch(false, s, lds, (uint8_t *)swizzled, rows, cols, stream);
}
