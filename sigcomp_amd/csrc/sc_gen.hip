// sc_gen.hip -- the codec for model architectures other than the bundled one
// (any window, embedding width, hidden width and layer count; the last layer
// gives 256 logits): the reference's GPU codec runs any shapes
// (quant_mlp_export.py:21-101,215-269), and its archives name their model
// dims (main.py:1086-1094).
//
// The specialised kernels keep everything of an evaluation on chip; here
// each stage is its own launch over a batch of rows in device memory:
//   k_gen_embed   token windows -> layer-0 input rows (zero padded to a
//                 multiple of 32 columns)
//   k_gen_linear  one quantised linear layer: v_mfma_i32_32x32x32_i8 over
//                 weights packed in fragment order (zero padded to 32 x 32
//                 tiles) and the rows from memory, then the per-channel
//                 requantisation of cpu_int_kernels.py:5-14 (64-bit form)
//   k_gen_pairs   logits -> (cumulative frequency, frequency) of each coded
//                 token, then the existing range encoder (k_encode_pairs)
//   k_gen_dec_*   one decoder step per chunk from its logits, the coder state
//                 in the caller's workspace
// Padded weight rows and columns are zero, so padded features requantise to
// zero and add nothing to the next layer.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <string>

#include "sc_fed.h"
#include "sc_gen.h"

namespace sc {
namespace {

// ---- embedding gather ----------------------------------------------------

enum GenSource { SRC_CTX = 0, SRC_TILES = 1, SRC_DECODE = 2 };

// Row r of the batch, window position p: the token, or SOS before the
// sequence start.  SRC_CTX: ctx[r * W + p] (int64, checked); SRC_TILES: row
// r is step t0 + i of the chunk whose step t0 is token `base` (tile
// descriptor r / 128 + tile0, i = r % 128), its context the tokens before it
// in the token array; SRC_DECODE: row r is chunk r at step t, its context
// the tokens it has decoded.
struct GenRows {
    int src;
    const int64_t *ctx;                 // SRC_CTX
    const uint8_t *tokens;              // SRC_TILES / SRC_DECODE
    const int4 *desc;                   // SRC_TILES
    int64_t tile0;
    const int32_t *tile_count;          // SRC_TILES: number of real tiles (device)
    const int64_t *tok_off;             // SRC_DECODE
    const int32_t *lengths;             // SRC_DECODE
    int32_t t;                          // SRC_DECODE
};

__device__ __forceinline__ int gen_token(const GenRows &g, int64_t r, int p, int W, bool &valid_row) {
    if (g.src == SRC_CTX) return (int)g.ctx[r * W + p];
    if (g.src == SRC_TILES) {
        const int64_t tile = g.tile0 + r / R_GEN_TILE;
        const int i = (int)(r % R_GEN_TILE);
        if (tile >= *g.tile_count) {
            valid_row = false;
            return SOS;
        }
        const int4 d = g.desc[tile];
        const int64_t base = (int64_t)(uint32_t)d.x | ((int64_t)d.y << 32);
        if (i >= d.z) valid_row = false;
        const int64_t s = (int64_t)d.w + i - W + p;   // sequence step of window position p
        return s < 0 || !valid_row ? SOS : (int)g.tokens[base + i - W + p];
    }
    const int64_t s = (int64_t)g.t - W + p;
    if (g.t >= g.lengths[r]) valid_row = false;
    return s < 0 || !valid_row ? SOS : (int)g.tokens[g.tok_off[r] + s];
}

// One thread per (row, window position): copies the token's embedding row
// (emb_dim bytes) into X[r][p * emb_dim ..]; the padding columns and rows
// past `rows` are zero.  Out-of-range context tokens set status[0].
__global__ __launch_bounds__(256) void k_gen_embed(const int8_t *__restrict__ emb, int32_t emb_dim, int32_t W,
                                                   GenRows g, int64_t rows, int64_t rows_p, int8_t *__restrict__ X,
                                                   int64_t ldx, int32_t *__restrict__ status) {
    const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t r = id / (W + 1);
    const int p = (int)(id % (W + 1));
    if (r >= rows_p) return;
    int8_t *row = X + r * ldx;
    if (p == W) {   // this thread clears the padding columns
        for (int64_t k = (int64_t)W * emb_dim; k < ldx; ++k) row[k] = 0;
        return;
    }
    bool valid = r < rows;
    int tok = valid ? gen_token(g, r, p, W, valid) : SOS;
    if (tok < 0 || tok > SOS) {
        if (status) status[0] = SC_STATUS_BAD_TOKEN;
        tok = 0;
    }
    const int8_t *e = emb + (int64_t)tok * emb_dim;
    int8_t *dst = row + (int64_t)p * emb_dim;
    for (int j = 0; j < emb_dim; ++j) dst[j] = r < rows ? e[j] : (int8_t)0;
}

// ---- one linear layer ----------------------------------------------------

// Y[r][n] = requant(sum_k W[n][k] X[r][k] + bias[n]) for rows r < rows of
// the 64-row block and the 64-feature block of the grid; wave w computes
// row tile w & 1, n-tile w >> 1 as one 32 x 32 MFMA tile (transposed:
// D[n][r], A = weight fragment, B = 16 bytes of row r).  X has rows_p
// rows of ldx bytes (ldx = the layer's k-tiles x 32).
__global__ __launch_bounds__(256) void k_gen_linear(LayerDev L, const int8_t *__restrict__ X, int64_t ldx,
                                                    int64_t rows, int8_t *__restrict__ Y, int64_t ldy) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t r0 = (int64_t)blockIdx.x * 64 + (wave & 1) * 32;
    const int nt = blockIdx.y * 2 + (wave >> 1);
    const int NT = (L.n + 31) / 32;
    if (nt >= NT) return;
    const int KT = L.kt;
    const v4i *wf = L.w + (int64_t)nt * KT * 64 + lane;
    const int8_t *xr = X + (r0 + (lane & 31)) * ldx + (lane >> 5) * 16;
    v16i acc = {};
    for (int kt = 0; kt < KT; ++kt) {
        const v4i a = wf[(int64_t)kt * 64];
        const v4i b = *(const v4i *)(xr + kt * 32);
        acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, acc, 0, 0, 0);
    }
    const uint32_t *par = L.par + (int64_t)nt * PAR_DWORDS;
    const int64_t r = r0 + (lane & 31);
    const int lo = L.relu ? 0 : -128;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int nl = 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
        const uint32_t sh = (par[64 + (nl >> 2)] >> (8 * (nl & 3))) & 0xFFu;
        const uint32_t q = requant_u8(acc[v], (int)par[nl], par[32 + nl], sh, lo);
        if (r < rows) Y[r * ldy + nt * 32 + nl] = (int8_t)(uint8_t)q;
    }
}

// ---- frequencies of the coded tokens (compress) -----------------------------

// 16 rows per workgroup (16-lane rows); row r = step of a tile as in
// k_gen_embed; its token's (cum, freq) go to pairs[token index].
__global__ __launch_bounds__(256) void k_gen_pairs(const int8_t *__restrict__ logits, int64_t rows,
                                                   const uint64_t *__restrict__ lut, const uint8_t *__restrict__ tokens,
                                                   const int4 *__restrict__ desc, int64_t tile0,
                                                   const int32_t *__restrict__ tile_count, uint2 *__restrict__ pairs) {
    __shared__ double s_lut[VOCAB];
    load_lut_lds(lut, s_lut);
    __syncthreads();
    const int u = threadIdx.x & 15;
    const int64_t r = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
    const v4i raw = r < rows ? *(const v4i *)(logits + r * VOCAB + 16 * u) : v4i{0, 0, 0, 0};
    Freq16 fr;
    row_frequencies16(raw, s_lut, u, fr);
    if (r >= rows) return;
    const int64_t tile = tile0 + r / R_GEN_TILE;
    const int i = (int)(r % R_GEN_TILE);
    if (tile >= *tile_count) return;
    const int4 d = desc[tile];
    if (i >= d.z) return;
    const int64_t g = ((int64_t)(uint32_t)d.x | ((int64_t)d.y << 32)) + i;
    const int s = tokens[g];
    if ((s >> 4) != u) return;   // the lane holding the symbol
    uint32_t cum, freq;
    freq16_at(fr, s & 15, cum, freq);
    pairs[g] = make_uint2(cum, freq);
}

// ---- decoder steps (decompress) ---------------------------------------------

// CpuRangeDecoder.__init__ (cpu_entropy_coding.py:466-474) for every chunk.
__global__ __launch_bounds__(256) void k_gen_dec_init(const uint32_t *__restrict__ words,
                                                      const int64_t *__restrict__ word_off,
                                                      const int32_t *__restrict__ word_cnt, int64_t n,
                                                      DecState *__restrict__ st) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n) return;
    const int32_t cnt = word_cnt[c];
    const uint32_t *w = words + word_off[c];
    const int take = cnt < 2 ? cnt : 2;
    uint64_t point = 0;
    for (int i = 0; i < take; ++i) point = (point << 32) | w[i];
    if (cnt == 1) point <<= 32;
    st[c] = DecState{0ull, ~0ull, point, take, 0, 0, 0};
}

// One decoder step at step t for every chunk with t < lengths[c] and a
// valid stream so far (_decode_partition, cpu_entropy_coding.py:230-266):
// 16 chunks per workgroup, the frequency rule on 16-lane rows.
__global__ __launch_bounds__(256) void k_gen_dec_step(const int8_t *__restrict__ logits, int64_t n,
                                                      const uint64_t *__restrict__ lut, int32_t t,
                                                      const int32_t *__restrict__ lengths,
                                                      const uint32_t *__restrict__ words,
                                                      const int64_t *__restrict__ word_off,
                                                      const int32_t *__restrict__ word_cnt,
                                                      uint8_t *__restrict__ tokens, const int64_t *__restrict__ tok_off,
                                                      DecState *__restrict__ st) {
    __shared__ double s_lut[VOCAB];
    load_lut_lds(lut, s_lut);
    __syncthreads();
    const int lane = threadIdx.x & 63, u = threadIdx.x & 15;
    const int64_t c = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
    const v4i raw = c < n ? *(const v4i *)(logits + c * VOCAB + 16 * u) : v4i{0, 0, 0, 0};
    Freq16 fr;
    row_frequencies16(raw, s_lut, u, fr);
    DecState d{0ull, ~0ull, 0ull, 0, 1, 0, 0};
    const bool active = c < n && t < lengths[c] && (d = st[c]).stat == 0;
    const uint64_t scale = d.range >> 24;
    uint32_t q = 0;
    const bool ok = scale != 0 && dec_quantile(d.point - d.lower, scale, q);
    uint32_t cum, freq;
    const int sym = dec_symbol16(fr, q, lane, cum, freq);
    if (!active || u != 0) return;
    if (!ok) {
        st[c].stat = SC_STATUS_INVALID_STREAM;
        return;
    }
    uint64_t lower = d.lower + mul_scale(scale, cum), range = mul_scale(scale, freq), point = d.point;
    int32_t rp = d.rpos;
    if (range < (1ull << 32)) {
        lower <<= 32;
        range <<= 32;
        point = (point << 32) | (rp < word_cnt[c] ? words[word_off[c] + rp] : 0u);
        rp += 1;
    }
    st[c] = DecState{lower, range, point, rp, 0, 0, 0};
    tokens[tok_off[c] + t] = (uint8_t)sym;
}

__global__ __launch_bounds__(256) void k_gen_dec_status(const DecState *__restrict__ st, int64_t n,
                                                        int32_t *__restrict__ status) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c < n) status[c] = st[c].stat;
}

// ---- the whole MLP of 32 rows in one workgroup ------------------------------
//
// Models whose activations fit the LDS (gen_fused_lds below: every width of
// a layer up to about 1,500, an embedding width that is a multiple of 16)
// run fused, but for few rows of wide ones (runs_fused below): a workgroup keeps 32 rows on chip from the token windows to the
// logits, streams each layer's weights once per 32 rows, and ends with what
// the call wants of the logits.  The decoder loops over its steps inside
// one launch.  One launch per stage cost seven launches a step (57 us for 64
// chunks of a 32 x 64 -> 256 -> 256 x 3 -> 256 model, of which 5 x 6.7 us the
// layers) and read every operand of every MFMA from memory.  Bound now by
// the CU's vector L1 (64 B/clock of weights).

enum GenOut { GEN_LOGITS = 0, GEN_CDF = 1, GEN_PAIRS = 2, GEN_DECODE = 3 };

constexpr int GEN_LDS = 156 * 1024;
constexpr int GEN_BLK = 8;          // k-tiles per block of a layer's loop
constexpr int GEN_MAX_WINDOW = 256;
// A compress call in separate launches against the fused one, beyond what
// their MLPs take (measured on seven models, 20 to 70 us)
constexpr int GEN_COMPRESS_US = 50;

// LDS of a fused workgroup, byte offsets (all multiples of 16)
struct GenLds {
    int32_t emb, emb_stride, ctx, slots, act[2], ld, logits, dec, bytes;
    uint32_t inv;   // ceil(2**20 / (emb_dim / 16)): 16-column chunk -> window position
};

// The rows' coder arrays of GEN_DECODE, after the common part
struct GenDecLds {
    static constexpr int SLOT = 0;
    static constexpr int LOWER = SLOT + WAVES * 2 * 4 * SLOT_DWORDS * 4;
    static constexpr int RANGE = LOWER + 32 * 8, POINT = RANGE + 32 * 8, WOFF = POINT + 32 * 8, TOFF = WOFF + 32 * 8;
    static constexpr int RPOS = TOFF + 32 * 8, WCNT = RPOS + 32 * 4, LEN = WCNT + 32 * 4, STAT = LEN + 32 * 4;
    static constexpr int WBASE = STAT + 32 * 4, WBUF_OFF = WBASE + 32 * 4, RING = WBUF_OFF + 32 * WBUF * 4;
    static constexpr int LAST = RING + 32 * WIN, MISC = LAST + 32 * 2, BYTES = MISC + 16;
};

struct GenArgs {
    const int64_t *ctx;            // GEN_LOGITS, GEN_CDF
    int8_t *logits;
    int32_t *cdf, *status;         // status: [1], or [n] in GEN_DECODE
    const uint8_t *tokens_in;      // GEN_PAIRS
    const int4 *desc;
    const int32_t *tile_count;
    uint2 *pairs;
    const uint32_t *words;         // GEN_DECODE
    const int64_t *word_off, *tok_off;
    const int32_t *word_cnt, *lengths;
    uint8_t *tokens;
    int64_t rows;                  // windows, tile descriptors (GEN_PAIRS) or chunks (GEN_DECODE)
};

// One layer for the workgroup's 32 rows: wave w computes n-tiles w, w + 4,
// ... two at a time (they share the operand fragments), GEN_BLK k-tiles per
// block with the next block's weights in flight.  `prep(kt0)` starts block
// kt0's operand reads, `frag(s)` is its fragment of k-tile kt0 + s.
template <class PrepFn, class FragFn>
__device__ __forceinline__ void gen_layer(const LayerDev &L, PrepFn prep, FragFn frag, uint8_t *out, int out_stride,
                                          int wave, int lane) {
    const int NT = (L.n + 31) / 32, KT = L.kt, g = lane >> 5, rl = lane & 31, voff = lane * 16;
    const int lo = L.relu ? 0 : -128;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)L.w, (short)0, L.bytes, 0x00020000);
    for (int nt = wave; nt < NT; nt += 2 * WAVES) {
        const bool two = nt + WAVES < NT;
        const int nb[2] = {nt, two ? nt + WAVES : nt};
        v4i w[2][GEN_BLK][2];
        auto load = [&](int kt0, v4i (&x)[GEN_BLK][2]) __attribute__((always_inline)) {
            // (beyond an n-tile: the next one's weights or the layer's last
            // fragment, which are not used)
#pragma unroll
            for (int s = 0; s < GEN_BLK; ++s)
#pragma unroll
                for (int j = 0; j < 2; ++j) x[s][j] = wload_s(rs, voff, min(nb[j] * KT + kt0 + s, NT * KT - 1) * 1024);
        };
        v16i acc[2] = {v16i{}, v16i{}};
        auto block = [&](int kt0, v4i (&cur)[GEN_BLK][2], v4i (&nxt)[GEN_BLK][2]) __attribute__((always_inline)) {
            if (kt0 + GEN_BLK < KT) load(kt0 + GEN_BLK, nxt);
            v4i b[GEN_BLK];
#pragma unroll
            for (int s = 0; s < GEN_BLK; ++s) b[s] = frag(kt0, s);
            auto products = [&](int s) __attribute__((always_inline)) {
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(cur[s][j], b[s], acc[j], 0, 0, 0);
            };
            // whole blocks in one run of instructions, the next block's
            // addresses beside the products (a branch per k-tile kept the
            // scheduler from mixing them: with it gone the bounded addresses of
            // the weight loads cost nothing, 5.28 -> 5.26 ms for the round
            // trip of 64 chunks x 256 tokens, 5.14 without the bound)
            if (kt0 + GEN_BLK <= KT) {
                prep(kt0 + GEN_BLK);
#pragma unroll
                for (int s = 0; s < GEN_BLK; ++s) products(s);
            } else {
#pragma unroll
                for (int s = 0; s < GEN_BLK; ++s)
                    if (kt0 + s < KT) products(s);
            }
        };
        prep(0);
        load(0, w[0]);
        // the requantisation's parameters behind the first weights
        v4i pb[2][4], pm[2][4];
        uint32_t ps[2][4];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {   // register 4 q + e: feature 8 q + 4 g + e
                const uint32_t *par = L.par + (int64_t)nb[j] * PAR_DWORDS + 8 * q + 4 * g;
                pb[j][q] = *(const v4i *)par;
                pm[j][q] = *(const v4i *)(par + 32);
                ps[j][q] = L.par[(int64_t)nb[j] * PAR_DWORDS + 64 + 2 * q + g];
            }
#pragma unroll 1
        for (int kt0 = 0; kt0 < KT; kt0 += 2 * GEN_BLK) {
            block(kt0, w[0], w[1]);
            if (kt0 + GEN_BLK < KT) block(kt0 + GEN_BLK, w[1], w[0]);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if (j == 1 && !two) break;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int nl = 8 * q + 4 * g;
                uint32_t pk = 0;
                // 32-bit high products where the whole layer allows them
                if (L.fast == LAYER_FAST_GENERIC) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        pk |= requant_u8_fast(acc[j][4 * q + e], pb[j][q][e], pm[j][q][e],
                                              ((ps[j][q] >> (8 * e)) & 0xFFu) - 32u, lo)
                              << (8 * e);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        pk |= requant_u8(acc[j][4 * q + e], pb[j][q][e], (uint32_t)pm[j][q][e], (ps[j][q] >> (8 * e)) & 0xFFu, lo)
                              << (8 * e);
                }
                *(uint32_t *)(out + rl * out_stride + nb[j] * 32 + nl) = pk;
            }
        }
    }
    __syncthreads();
}

// The MLP: layer 0's operands gathered from the embedding table in LDS by the
// tokens of slot((position)), the others from the activation buffers; logits
// at P.logits, PACT_ROW bytes per row.
template <class SlotFn>
__device__ __forceinline__ void gen_mlp_rows(const ModelDev &M, const GenLds &P, uint8_t *s_mem, SlotFn slot, int wave,
                                             int lane) {
    const int g = lane >> 5, rl = lane & 31, E = M.emb_dim, W = M.window;
    const uint8_t *s_emb = s_mem + P.emb;
    const uint16_t *s_ctx = (const uint16_t *)(s_mem + P.ctx);
    for (int l = 0; l < M.n_layers; ++l) {
        const LayerDev &L = M.layer[l];
        const bool last = l == M.n_layers - 1;
        uint8_t *out = s_mem + (last ? P.logits : P.act[l & 1]);
        const int stride = last ? PACT_ROW : P.ld;
        if (l == 0) {
            int addr[GEN_BLK];
            gen_layer(
                L,
                [&](int kt0) __attribute__((always_inline)) {
#pragma unroll
                    for (int s = 0; s < GEN_BLK; ++s) {
                        // 16 columns of one position (E is a multiple of 16);
                        // columns past the window have zero weights
                        // (exact while ch * (E / 16) < 2**20: the windows and widths
                        // that fit the LDS reach 174,000)
                        const int ch = (kt0 + s) * 2 + g, p = min((int)(((uint32_t)ch * P.inv) >> 20), W - 1);
                        addr[s] = (int)s_ctx[slot(p) * 32 + rl] * P.emb_stride + min(ch * 16 - p * E, E - 16);
                    }
                },
                [&](int, int s) __attribute__((always_inline)) { return *(const v4i *)(s_emb + addr[s]); }, out, stride,
                wave, lane);
        } else {
            const uint8_t *in = s_mem + P.act[(l - 1) & 1] + rl * P.ld + 16 * g;
            gen_layer(
                L, [](int) {},
                [&](int kt0, int s) __attribute__((always_inline)) {
                    return *(const v4i *)(in + min(kt0 + s, L.kt - 1) * 32);
                },
                out, stride, wave, lane);
        }
    }
}

template <int OUT>
__global__ __launch_bounds__(THREADS, 1) void k_gen_fused(ModelDev M, GenLds P, GenArgs A) {
    __shared__ __attribute__((aligned(16))) uint8_t s_mem[GEN_LDS];
    __shared__ double s_lut[VOCAB];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int u = lane & 15, q4 = lane >> 4, W = M.window, E = M.emb_dim;
    uint16_t *s_ctx = (uint16_t *)(s_mem + P.ctx);   // [slot][row]
    const uint8_t *s_log = s_mem + P.logits;
    for (int i = threadIdx.x; i < EMB_ROWS * (E / 16); i += THREADS) {
        const int tok = i / (E / 16), ch = i % (E / 16);
        *(v4i *)(s_mem + P.emb + tok * P.emb_stride + ch * 16) = *(const v4i *)(M.emb + tok * E + ch * 16);
    }
    load_lut_lds(M.lut, s_lut);
    if constexpr (OUT != GEN_DECODE) {
        const int64_t tiles = OUT == GEN_PAIRS ? min<int64_t>(*A.tile_count, A.rows) * (R_GEN_TILE / 32) : (A.rows + 31) / 32;
        for (int64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
            const int64_t r0 = tile * 32;
            int4 d{};
            int64_t base = 0;
            int i0 = 0, valid = 32;
            if constexpr (OUT == GEN_PAIRS) {
                d = A.desc[tile / (R_GEN_TILE / 32)];
                base = (int64_t)(uint32_t)d.x | ((int64_t)d.y << 32);
                i0 = (int)(tile % (R_GEN_TILE / 32)) * 32;
                valid = min(32, d.z - i0);
                if (valid <= 0) continue;   // (the whole workgroup)
            } else {
                valid = (int)min<int64_t>(32, A.rows - r0);
            }
            __syncthreads();
            for (int i = threadIdx.x; i < 32 * W; i += THREADS) {
                const int r = i / W, p = i % W;
                int tok = SOS;
                if constexpr (OUT == GEN_PAIRS) {
                    const int64_t at = (int64_t)i0 + r - W + p;   // step relative to the tile's first
                    if (r < valid && d.w + at >= 0) tok = A.tokens_in[base + at];
                } else if (r < valid) {
                    const int64_t v = A.ctx[(r0 + r) * W + p];
                    const bool ok = (uint64_t)v <= (uint64_t)SOS;
                    if (!ok) A.status[0] = SC_STATUS_BAD_TOKEN;
                    tok = ok ? (int)v : 0;
                }
                s_ctx[p * 32 + r] = (uint16_t)tok;
            }
            __syncthreads();
            gen_mlp_rows(M, P, s_mem, [](int p) { return p; }, wave, lane);
            if constexpr (OUT == GEN_LOGITS) {
                for (int i = threadIdx.x; i < 32 * 16; i += THREADS) {
                    const int r = i >> 4, ch = i & 15;
                    if (r < valid) *(v4i *)(A.logits + (r0 + r) * VOCAB + ch * 16) = *(const v4i *)(s_log + pact_off(r, ch));
                }
            } else {
                for (int gi = wave; gi * 4 < valid; gi += WAVES) {
                    const int r = gi * 4 + q4;
                    Freq16 fr;
                    row_frequencies16(*(const v4i *)(s_log + pact_off(r, u)), s_lut, u, fr);
                    if (r >= valid) continue;
                    if constexpr (OUT == GEN_CDF) {
                        int32_t *dst = A.cdf + (r0 + r) * (VOCAB + 1) + 16 * u;
                        uint32_t c = fr.ex;
#pragma unroll
                        for (int k = 0; k < 16; ++k) {
                            dst[k] = (int32_t)c;
                            c += fr.f[k];
                        }
                        if (u == 15) dst[16] = (int32_t)TOTAL;
                    } else {
                        const int sym = A.tokens_in[base + i0 + r];
                        if ((sym >> 4) == u) {
                            uint32_t cum, freq;
                            freq16_at(fr, sym & 15, cum, freq);
                            A.pairs[base + i0 + r] = make_uint2(cum, freq);
                        }
                    }
                }
            }
        }
    } else {
        using D = GenDecLds;
        uint8_t *dec = s_mem + P.dec;
        int32_t *s_steps = (int32_t *)(dec + D::MISC);
        const FedRows c{s_log,
                        s_lut,
                        (uint64_t *)(dec + D::LOWER),
                        (uint64_t *)(dec + D::RANGE),
                        (uint64_t *)(dec + D::POINT),
                        (int64_t *)(dec + D::WOFF),
                        (int64_t *)(dec + D::TOFF),
                        (int32_t *)(dec + D::RPOS),
                        (int32_t *)(dec + D::WCNT),
                        (int32_t *)(dec + D::LEN),
                        (int32_t *)(dec + D::STAT),
                        (int32_t *)(dec + D::WBASE),
                        (uint32_t *)(dec + D::WBUF_OFF),
                        dec + D::RING,
                        (uint16_t *)(dec + D::LAST)};
        uint32_t *slots = (uint32_t *)(dec + D::SLOT) + wave * (2 * 4 * SLOT_DWORDS);
        const int64_t c0 = (int64_t)blockIdx.x * 32;
        if (threadIdx.x == 0) *s_steps = 0;
        for (int i = threadIdx.x; i < 32 * P.slots; i += THREADS) s_ctx[i] = SOS;
        __syncthreads();
        if (threadIdx.x < 32) {
            const int r = threadIdx.x;
            const int64_t ch = c0 + r;
            const bool in = ch < A.rows;
            const int32_t len = in ? A.lengths[ch] : 0, cnt = in ? A.word_cnt[ch] : 0;
            const int64_t woff = in ? A.word_off[ch] : 0;
            int take;
            c.point[r] = dec_init_point(A.words + woff, cnt, take);
            c.lower[r] = 0ull;
            c.range[r] = ~0ull;
            c.rpos[r] = take;
            c.stat[r] = 0;
            c.wcnt[r] = cnt;
            c.woff[r] = woff;
            c.toff[r] = in ? A.tok_off[ch] : 0;
            c.len[r] = len;
            atomicMax(s_steps, len);
        }
        for (int i = threadIdx.x; i < 32 * WIN / 4; i += THREADS) ((uint32_t *)c.ring)[i] = 0;
        __syncthreads();
        const int32_t steps = *s_steps;
        auto refill = [&] {   // the next 64 words of every row
            for (int r = wave; r < 32; r += WAVES) {
                const int32_t at = c.rpos[r], cnt = c.wcnt[r];
                c.wbuf[r * WBUF + lane] = at + lane < cnt ? A.words[c.woff[r] + at + lane] : 0u;
                if (lane == 0) c.wbase[r] = at;
            }
        };
        refill();
        __syncthreads();
        const int mask = P.slots - 1;   // the window's ring has a power of two slots
#pragma unroll 1
        for (int32_t t = 0; t < steps; ++t) {
            gen_mlp_rows(M, P, s_mem, [&](int p) { return (t - W + p) & mask; }, wave, lane);
            for (int gi = wave; gi < 8; gi += 2 * WAVES) {
                const int ra = gi * 4 + q4, rb = ra + 4 * WAVES;
                const bool a = __builtin_amdgcn_ballot_w64(t < c.len[ra] && c.stat[ra] == 0) != 0;
                const bool b = __builtin_amdgcn_ballot_w64(t < c.len[rb] && c.stat[rb] == 0) != 0;
                if (a && b) fed_decode_rows<2>(c, slots, t, gi, lane);
                else if (a) fed_decode_rows<1>(c, slots, t, gi, lane);
                else if (b) fed_decode_rows<1>(c, slots, t, gi + WAVES, lane);
            }
            __syncthreads();
            if (threadIdx.x < 32) s_ctx[(t & mask) * 32 + threadIdx.x] = c.ring[threadIdx.x * WIN + (t & (WIN - 1))];
            if ((t & (WIN - 1)) == WIN - 1 || t == steps - 1) {
                const int32_t p = (t & ~(WIN - 1)) + lane;
                for (int r = wave; r < 32; r += WAVES)
                    if (p <= t && p < c.len[r]) A.tokens[c.toff[r] + p] = c.ring[r * WIN + lane];
                refill();
            }
            __syncthreads();
        }
        if (threadIdx.x < 32 && c0 + threadIdx.x < A.rows) A.status[c0 + threadIdx.x] = c.stat[threadIdx.x];
    }
}

// ---- logits -> int32 CDF (sc_mlp_forward_cdf) ------------------------------

__global__ __launch_bounds__(256) void k_gen_cdf32(const int8_t *__restrict__ logits, int64_t rows,
                                                   const uint64_t *__restrict__ lut, int32_t *__restrict__ cdf) {
    __shared__ double s_lut[VOCAB];
    load_lut_lds(lut, s_lut);
    __syncthreads();
    const int u = threadIdx.x & 15;
    const int64_t r = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
    const v4i raw = r < rows ? *(const v4i *)(logits + r * VOCAB + 16 * u) : v4i{0, 0, 0, 0};
    Freq16 fr;
    row_frequencies16(raw, s_lut, u, fr);
    if (r >= rows) return;
    int32_t *dst = cdf + r * (VOCAB + 1) + 16 * u;
    uint32_t c = fr.ex;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        dst[k] = (int32_t)c;
        c += fr.f[k];
    }
    if (u == 15) dst[16] = (int32_t)TOTAL;
}

// ---- host side -------------------------------------------------------------

int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }

// The fused kernel's LDS for a model; bytes = 0 when it does not fit.
GenLds gen_fused_lds(const ModelDev &M) {
    GenLds P{};
    if (M.emb_dim % 16 || M.window > GEN_MAX_WINDOW) return P;
    P.slots = 1;
    while (P.slots < M.window) P.slots *= 2;
    int64_t ld = 0;   // activation rows: the widest hidden layer and a 16-byte pad (bank spread)
    for (int i = 0; i + 1 < M.n_layers; ++i) ld = std::max<int64_t>(ld, round_up(M.layer[i].n, 32) + 16);
    P.emb_stride = M.emb_dim + 16;
    P.inv = ((1u << 20) + M.emb_dim / 16 - 1) / (M.emb_dim / 16);
    int64_t at = 0;
    auto take = [&](int64_t bytes) {
        const int64_t o = at;
        at += round_up(bytes, 16);
        return o;
    };
    P.emb = (int32_t)take((int64_t)EMB_ROWS * P.emb_stride);
    P.ctx = (int32_t)take((int64_t)P.slots * 64);
    P.ld = (int32_t)std::min<int64_t>(ld, GEN_LDS);
    P.act[0] = (int32_t)take(32 * (int64_t)P.ld);
    P.act[1] = (int32_t)take(32 * (int64_t)P.ld);
    P.logits = (int32_t)take(32 * PACT_ROW);
    P.dec = (int32_t)take(GenDecLds::BYTES);
    P.bytes = at <= GEN_LDS && ld <= GEN_LDS ? (int32_t)at : 0;
    return P;
}

int n_cu() {
    int dev = 0, cu = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        cu = 256;
    return std::max(cu, 1);
}

// Workgroups of a fused launch over `tiles` 32-row tiles: one per CU.
unsigned fused_grid(int64_t tiles) { return (unsigned)std::max<int64_t>(1, std::min<int64_t>(tiles, n_cu())); }

// Whether a call whose MLP takes `rows` rows at a time runs fused.  A fused
// workgroup streams all weights through its CU (88 GB/s) for its 32 rows; the
// separate launches spread a layer's n-tiles over the device, but each waits
// for its k-tiles one after the other and their rows go through memory.  So
// few rows of a model with wide layers are cheaper in separate launches:
// 16 chunks of a 64 x 128 -> 1024 x 6 -> 256 model take 138 us a step so and
// 188 fused, of a 64 x 16 -> 1400 x 4 -> 256 model 61 and 132; 4,096 chunks
// 797 and 183, 198 and 126.  The costs in us are least-squares fits to the
// decode steps of eighteen models (82 thousand to 14 million weights) at 1
// to 4,096 chunks, of which they choose the faster form every time.
// `once_us` is what the call's first separate launches cost beyond a step.
// SC_HIP_GEN_FUSED = 0 or 1 forces one form (comparisons and tests of both).
bool runs_fused(const ModelDev &M, const GenLds &P, int64_t rows, int once_us) {
    if (!P.bytes) return false;
    const char *env = getenv("SC_HIP_GEN_FUSED");
    if (env && (env[0] == '0' || env[0] == '1') && env[1] == 0) return env[0] == '1';
    double kts = 0, weights = 0, passes = 0, streamed = 0;
    for (int i = 0; i < M.n_layers; ++i) {
        // (a wave streams two n-tiles per pass, whether or not it has two)
        const int nt = (M.layer[i].n + 31) / 32, ps = (nt + 2 * WAVES - 1) / (2 * WAVES);
        kts += M.layer[i].kt;
        weights += (double)nt * M.layer[i].kt * 1024;
        passes += ps;
        streamed += (double)ps * 2 * WAVES * M.layer[i].kt * 1024;
    }
    const int64_t tiles = (rows + 31) / 32, cu = n_cu();
    const double fused = (double)((tiles + cu - 1) / cu) * (1.7 + 0.35 * M.n_layers + 1.32 * passes + streamed / 88.2e3);
    const double separate = once_us + 2.51 * (M.n_layers + 2) + 0.206 * kts + 0.192 * M.emb_dim +
                            (double)rows * ((double)M.window * M.emb_dim / 195e3 + weights / 379e6);
    return fused <= separate;
}

// Widest padded layer input / output of the model (bytes per row).
int64_t max_width(const ModelDev &M) {
    int64_t w = round_up((int64_t)M.window * M.emb_dim, 32);
    for (int i = 0; i < M.n_layers; ++i) w = std::max<int64_t>(w, round_up(M.layer[i].n, 32));
    return w;
}

// Rows per batch of a call that needs `needed` rows: at most
// GEN_BATCH_ROWS, at most what GEN_SCRATCH_BYTES holds at this model's width
// (two activation buffers and the logits per row), and no more than the
// call needs; a multiple of `unit` (64-row MLP tiles, 128-step compress
// tiles).  The widest model sc_model_create accepts (2**20 inputs) still
// gets 384 rows.
int64_t batch_rows(const ModelDev &M, int64_t needed, int64_t unit) {
    const int64_t per_row = 2 * max_width(M) + VOCAB;
    const int64_t fit = std::max<int64_t>(GEN_SCRATCH_BYTES / per_row / unit, 1) * unit;
    return std::min({GEN_BATCH_ROWS / unit * unit, fit, round_up(std::max<int64_t>(needed, 1), unit)});
}

hipError_t launch_check() { return hipGetLastError(); }

int fused_result(const char *what, std::string &err) {
    const hipError_t e = launch_check();
    if (e == hipSuccess) return SC_OK;
    err = std::string(what) + hipGetErrorString(e);
    return SC_ERR_HIP;
}

// Stream-ordered scratch of one call (hipMallocAsync / hipFreeAsync).
struct Scratch {
    void *p = nullptr;
    hipStream_t s;
    explicit Scratch(hipStream_t st) : s(st) {}
    hipError_t alloc(size_t bytes) { return hipMallocAsync(&p, bytes, s); }
    ~Scratch() {
        if (p) (void)hipFreeAsync(p, s);
    }
};

// The MLP over `rows` rows from `g` -> int8 logits [rows][256] at `logits`
// (row stride 256).  X0 / X1: ping-pong buffers of rows_p x max_width bytes.
hipError_t gen_mlp(const ModelDev &M, const GenRows &g, int64_t rows, int8_t *X0, int8_t *X1, int8_t *logits,
                   int32_t *status, hipStream_t s) {
    const int64_t rows_p = round_up(std::max<int64_t>(rows, 1), 64);
    const int W = M.window;
    const int64_t k0p = round_up((int64_t)W * M.emb_dim, 32);
    const int64_t threads = rows_p * (W + 1);
    hipLaunchKernelGGL(k_gen_embed, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, M.emb, M.emb_dim, W,
                       g, rows, rows_p, X0, k0p, status);
    hipError_t e = launch_check();
    if (e != hipSuccess) return e;
    int8_t *src = X0, *dst = X1;
    int64_t ld = k0p;
    for (int l = 0; l < M.n_layers; ++l) {
        const LayerDev &L = M.layer[l];
        const bool last = l == M.n_layers - 1;
        const int64_t ldy = last ? VOCAB : round_up(L.n, 32);
        int8_t *out = last ? logits : dst;
        const dim3 grid((unsigned)(rows_p / 64), (unsigned)((L.n + 63) / 64));
        hipLaunchKernelGGL(k_gen_linear, grid, dim3(256), 0, s, L, src, ld, last ? rows : rows_p, out, ldy);
        if ((e = launch_check()) != hipSuccess) return e;
        std::swap(src, dst);
        ld = ldy;
    }
    return hipSuccess;
}

}  // namespace

int gen_mlp_forward(const ModelDev &M, const int64_t *ctx, int64_t rows, int8_t *logits, int32_t *cdf,
                    int32_t *status, hipStream_t s, std::string &err) {
    if (const GenLds P = gen_fused_lds(M); runs_fused(M, P, rows, 0)) {
        GenArgs A{};
        A.ctx = ctx;
        A.logits = logits;
        A.cdf = cdf;
        A.status = status;
        A.rows = rows;
        hipLaunchKernelGGL(cdf ? k_gen_fused<GEN_CDF> : k_gen_fused<GEN_LOGITS>, dim3(fused_grid((rows + 31) / 32)),
                           dim3(THREADS), 0, s, M, P, A);
        return fused_result("generic MLP launch: ", err);
    }
    const int64_t B = batch_rows(M, rows, 64);
    const int64_t width = max_width(M), rows_p = B;
    Scratch scr(s);
    hipError_t e = scr.alloc((size_t)(2 * rows_p * width + (cdf ? rows_p * VOCAB : 0)));
    if (e != hipSuccess) {
        err = std::string("hipMallocAsync: ") + hipGetErrorString(e);
        return SC_ERR_HIP;
    }
    int8_t *X0 = (int8_t *)scr.p, *X1 = X0 + rows_p * width, *lg = X1 + rows_p * width;
    for (int64_t r0 = 0; r0 < rows; r0 += B) {
        const int64_t n = std::min(B, rows - r0);
        GenRows g{SRC_CTX, ctx + r0 * M.window, nullptr, nullptr, 0, nullptr, nullptr, nullptr, 0};
        int8_t *out = cdf ? lg : logits + r0 * VOCAB;
        if ((e = gen_mlp(M, g, n, X0, X1, out, status, s)) != hipSuccess) break;
        if (cdf) {
            hipLaunchKernelGGL(k_gen_cdf32, dim3((unsigned)((n + 15) / 16)), dim3(256), 0, s, lg, n, M.lut,
                               cdf + r0 * (VOCAB + 1));
            if ((e = launch_check()) != hipSuccess) break;
        }
    }
    if (e != hipSuccess) {
        err = std::string("generic MLP launch: ") + hipGetErrorString(e);
        return SC_ERR_HIP;
    }
    return SC_OK;
}

int gen_compress(const ModelDev &M, const uint8_t *tokens, const int32_t *tile_start, int64_t n_chunks,
                 const int4 *desc, int64_t max_tiles, uint2 *pairs, hipStream_t s, std::string &err) {
    if (const GenLds P = gen_fused_lds(M); runs_fused(M, P, max_tiles * R_GEN_TILE, GEN_COMPRESS_US)) {
        GenArgs A{};
        A.tokens_in = tokens;
        A.desc = desc;
        A.tile_count = tile_start + n_chunks;
        A.pairs = pairs;
        A.rows = max_tiles;
        hipLaunchKernelGGL(k_gen_fused<GEN_PAIRS>, dim3(fused_grid(max_tiles * (R_GEN_TILE / 32))), dim3(THREADS), 0, s, M,
                           P, A);
        return fused_result("generic compress launch: ", err);
    }
    const int64_t rows_b = batch_rows(M, max_tiles * R_GEN_TILE, R_GEN_TILE), width = max_width(M);
    const int64_t tiles_per = rows_b / R_GEN_TILE;
    Scratch scr(s);
    hipError_t e = scr.alloc((size_t)(2 * rows_b * width + rows_b * VOCAB));
    if (e != hipSuccess) {
        err = std::string("hipMallocAsync: ") + hipGetErrorString(e);
        return SC_ERR_HIP;
    }
    int8_t *X0 = (int8_t *)scr.p, *X1 = X0 + rows_b * width, *lg = X1 + rows_b * width;
    const int32_t *count = tile_start + n_chunks;   // tiles of the call (device)
    for (int64_t t0 = 0; t0 < max_tiles && e == hipSuccess; t0 += tiles_per) {
        const int64_t rows = std::min(tiles_per, max_tiles - t0) * R_GEN_TILE;
        GenRows g{SRC_TILES, nullptr, tokens, desc, t0, count, nullptr, nullptr, 0};
        if ((e = gen_mlp(M, g, rows, X0, X1, lg, nullptr, s)) != hipSuccess) break;
        hipLaunchKernelGGL(k_gen_pairs, dim3((unsigned)((rows + 15) / 16)), dim3(256), 0, s, lg, rows, M.lut, tokens,
                           desc, t0, count, pairs);
        e = launch_check();
    }
    if (e != hipSuccess) {
        err = std::string("generic compress launch: ") + hipGetErrorString(e);
        return SC_ERR_HIP;
    }
    return SC_OK;
}

int gen_decompress(const ModelDev &M, const uint32_t *words, const int64_t *word_off, const int32_t *word_cnt,
                   const int32_t *lengths, int64_t n_chunks, uint8_t *tokens, const int64_t *tok_off,
                   int32_t *status, DecState *state, int32_t max_len, hipStream_t s, std::string &err) {
    if (const GenLds P = gen_fused_lds(M); runs_fused(M, P, n_chunks, 0)) {
        GenArgs A{};
        A.status = status;
        A.words = words;
        A.word_off = word_off;
        A.word_cnt = word_cnt;
        A.lengths = lengths;
        A.tokens = tokens;
        A.tok_off = tok_off;
        A.rows = n_chunks;
        hipLaunchKernelGGL(k_gen_fused<GEN_DECODE>, dim3((unsigned)((n_chunks + 31) / 32)), dim3(THREADS), 0, s, M, P, A);
        return fused_result("generic decompress launch: ", err);
    }
    const int64_t width = max_width(M);
    const int64_t B = batch_rows(M, n_chunks, 64), rows_p = B;
    Scratch scr(s);
    hipError_t e = scr.alloc((size_t)(2 * rows_p * width + rows_p * VOCAB));
    if (e != hipSuccess) {
        err = std::string("hipMallocAsync: ") + hipGetErrorString(e);
        return SC_ERR_HIP;
    }
    int8_t *X0 = (int8_t *)scr.p, *X1 = X0 + rows_p * width, *lg = X1 + rows_p * width;
    // groups of at most B chunks, each decoded step by step
    for (int64_t c0 = 0; c0 < n_chunks && e == hipSuccess; c0 += B) {
        const int64_t n = std::min(B, n_chunks - c0);
        hipLaunchKernelGGL(k_gen_dec_init, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, words, word_off + c0,
                           word_cnt + c0, n, state + c0);
        if ((e = launch_check()) != hipSuccess) break;
        for (int32_t t = 0; t < max_len && e == hipSuccess; ++t) {
            GenRows g{SRC_DECODE, nullptr, tokens, nullptr, 0, nullptr, tok_off + c0, lengths + c0, t};
            if ((e = gen_mlp(M, g, n, X0, X1, lg, nullptr, s)) != hipSuccess) break;
            hipLaunchKernelGGL(k_gen_dec_step, dim3((unsigned)((n + 15) / 16)), dim3(256), 0, s, lg, n, M.lut, t,
                               lengths + c0, words, word_off + c0, word_cnt + c0, tokens, tok_off + c0, state + c0);
            e = launch_check();
        }
        if (e != hipSuccess) break;
        hipLaunchKernelGGL(k_gen_dec_status, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, state + c0, n,
                           status + c0);
        e = launch_check();
    }
    if (e != hipSuccess) {
        err = std::string("generic decompress launch: ") + hipGetErrorString(e);
        return SC_ERR_HIP;
    }
    return SC_OK;
}

}  // namespace sc
