// sc_ctx_two.hip -- explicit context windows, few rows: layer 0 spread over
// the chip, then the rest per 32 rows.
//
// A call of up to a few thousand rows leaves most CUs idle, and each 32-row
// tile streams the 6.2 MB model through one CU (63 us).  Here layer 0 (4.2 MB
// of it) runs as one workgroup per n-tile and 32 rows, its four waves over a
// quarter of the window each, and hands its requantised features (512 bytes
// per row, hidden order) to a second launch that streams the other 2 MB per
// 32 rows.  The first launch is bound by its weight slab (256 KB per
// workgroup) and the staging of its tables, the second by its CU's vector L1.
#include "sc_kernels.h"

namespace sc {
namespace {

constexpr int CTX_POS = WIN / WAVES;   // window positions per wave

__global__ __launch_bounds__(THREADS, 2) void k_ctx_layer0(ModelDev M, const int64_t *__restrict__ ctx, int64_t rows,
                                                           uint8_t *__restrict__ feat, int32_t *__restrict__ status) {
    __shared__ __attribute__((aligned(16))) uint8_t s_emb[EMB_BYTES];
    constexpr int CTX_STRIDE = WIN + 2;   // (as k_mlp_context: 32 rows' halfwords in different banks)
    __shared__ __attribute__((aligned(16))) uint16_t s_ctx[32 * CTX_STRIDE];
    __shared__ __attribute__((aligned(16))) v4i s_red[WAVES * 4 * 64];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    // consecutive workgroups take consecutive n-tiles: each XCD's L2 sees two
    // of the sixteen slabs
    const int nt = (int)(blockIdx.x % (HID / 32));
    const int64_t row0 = (int64_t)(blockIdx.x / (HID / 32)) * 32;
    constexpr int PER = 32 * WIN / THREADS;
    const int64_t *src = ctx + row0 * WIN + threadIdx.x;
    const int64_t lim = rows - row0 - wave;   // element j is row 4j + wave, position lane
    int64_t v[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) v[j] = 4 * j < lim ? src[j * THREADS] : 0;
    load_emb_lds(M.emb, s_emb);
    int bad = 0;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const bool ok = (uint64_t)v[j] <= (uint64_t)SOS;
        bad |= !ok;
        s_ctx[(4 * j + wave) * CTX_STRIDE + lane] = (uint16_t)emb_off(ok ? (int)v[j] : 0, 0);
    }
    if (bad) status[0] = SC_STATUS_BAD_TOKEN;
    __syncthreads();
    const LayerDev &L = M.layer[0];
    const v16i zero = {};
    const v16i acc = gemm_layer0_one<CTX_POS, CTX_POS>(
        make_wstream(L.w, L.bytes), nt, wave * CTX_POS, s_emb, [&](int r, int p) { return (int)s_ctx[r * CTX_STRIDE + p]; },
        zero, lane);
#pragma unroll
    for (int e = 0; e < 4; ++e)
        s_red[(wave * 4 + e) * 64 + lane] = v4i{acc[4 * e], acc[4 * e + 1], acc[4 * e + 2], acc[4 * e + 3]};
    __syncthreads();
    // wave w: registers 4 w .. + 3 of the tile = features 8 w + 4 g + e
    const int g = lane >> 5, rl = lane & 31;
    v4i x = s_red[wave * 64 + lane];
#pragma unroll
    for (int f = 1; f < WAVES; ++f) {
        const v4i y = s_red[(f * 4 + wave) * 64 + lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = (int)((uint32_t)x[e] + (uint32_t)y[e]);
    }
    const uint32_t *par = L.par + nt * PAR_DWORDS;
    const int n = 8 * wave + 4 * g;
    const uint32_t sh = par[64 + (n >> 2)];
    uint32_t pk = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e)   // (ReLU: the pipelined cores' layer 0)
        pk |= requant_u8_fast(x[e], (int)par[n + e], (int)par[32 + n + e], (sh >> (8 * e)) & 63u, 0) << (8 * e);
    *(uint32_t *)(feat + (row0 + rl) * HID + (nt * 2 + g) * 16 + 4 * wave) = pk;
}

template <int MODE, bool UNI>
__global__ __launch_bounds__(THREADS, 1) void k_ctx_rest(ModelDev M, const uint8_t *__restrict__ feat, int64_t rows,
                                                         int8_t *__restrict__ logits, int32_t *__restrict__ cdf) {
    constexpr int RT = 1, PPD = ppd<RT>();
    __shared__ __attribute__((aligned(16))) uint8_t s_act[32 * PACT_ROW];
    __shared__ __attribute__((aligned(16))) uint32_t s_par[pipe_par_dwords<UNI>()];
    __shared__ double s_lut[VOCAB];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int nb0 = 2 * wave;
    const int64_t row0 = (int64_t)blockIdx.x * 32;
    uint32_t *s_parw = s_par + wave * PIPE_SLOTS * Slot<UNI>::BLK;
    v16i accA[PNT][RT], accB[PNT][RT];
    v4i w[2][PPD][PNT];
    uint32_t pk[PNT][RT][4];
    {
        const __amdgpu_buffer_rsrc_t rs1 = layer_rsrc(M.layer[1]);
#pragma unroll
        for (int s = 0; s < PPD; ++s)
#pragma unroll
            for (int j = 0; j < PNT; ++j) w[0][s][j] = wload_s(rs1, lane * 16, ((nb0 + j) * KTH + s) * 1024);
        uint32_t prn[Slot<UNI>::LANE];
        par_fetch<UNI>(M.layer[1].par, nb0, lane, prn);
        par_put<UNI>(s_parw + slot_p0(1) * Slot<UNI>::BLK, prn, lane);
    }
    // (whole tiles of features: the first launch writes 32 rows)
    constexpr int PER = 32 * (HID / 16) / THREADS;
    v4i f[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) f[j] = *(const v4i *)(feat + row0 * HID + (j * THREADS + threadIdx.x) * 16);
    load_lut_lds(M.lut, s_lut);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int i = j * THREADS + threadIdx.x;
        *(v4i *)(s_act + pact_off(i / (HID / 16), i % (HID / 16))) = f[j];
    }
    __syncthreads();
    const int last = M.n_layers - 1;
    if (last == 1) {
        pipe_hidden<RT, true, UNI, true>(M.layer[0], M.layer[1], M.layer[1], s_act, s_parw, 1, accA, accB, w, pk, wave,
                                         lane);
    } else {
        pipe_hidden<RT, false, UNI, true>(M.layer[0], M.layer[1], M.layer[2], s_act, s_parw, 1, accA, accB, w, pk, wave,
                                          lane);
#pragma unroll 1
        for (int l = 2; l < last; ++l)
            pipe_hidden<RT, false, UNI>(M.layer[l - 1], M.layer[l], M.layer[l + 1], s_act, s_parw, l, accA, accB, w, pk,
                                        wave, lane);
        pipe_hidden<RT, true, UNI>(M.layer[last - 1], M.layer[last], M.layer[last], s_act, s_parw, last, accA, accB, w,
                                   pk, wave, lane);
    }
    const int valid = (int)min<int64_t>(32, rows - row0);
    if constexpr (MODE == OUT_LOGITS) {
        for (int i = threadIdx.x; i < 32 * 16; i += THREADS) {
            const int r = i >> 4, c = i & 15;
            if (r < valid) *(v4i *)(logits + (row0 + r) * VOCAB + c * 16) = *(const v4i *)(s_act + pact_off(r, c));
        }
    } else {
        const int u = lane & 15;
        for (int gi = wave; gi * 4 < valid; gi += WAVES) {
            const int r = gi * 4 + (lane >> 4);
            Freq16 fr;
            row_frequencies16(*(const v4i *)(s_act + pact_off(r, u)), s_lut, u, fr);
            if (r >= valid) continue;
            int32_t *dst = cdf + (row0 + r) * (VOCAB + 1) + 16 * u;
            uint32_t c = fr.ex;
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                dst[k] = (int32_t)c;
                c += fr.f[k];
            }
            if (u == 15) dst[16] = (int32_t)TOTAL;
        }
    }
}

}  // namespace

void launch_ctx_two(const ModelDev &M, hipStream_t s, const int64_t *ctx, int64_t rows, int8_t *logits, int32_t *cdf,
                    int32_t *status, uint8_t *feat) {
    const unsigned tiles = (unsigned)((rows + 31) / 32);
    hipLaunchKernelGGL(k_ctx_layer0, dim3(tiles * (HID / 32)), dim3(THREADS), 0, s, M, ctx, rows, feat, status);
    const bool uni = M.pipe == CORE_PIPE_UNI;
    auto *rest = logits ? (uni ? k_ctx_rest<OUT_LOGITS, true> : k_ctx_rest<OUT_LOGITS, false>)
                        : (uni ? k_ctx_rest<OUT_CDF32, true> : k_ctx_rest<OUT_CDF32, false>);
    hipLaunchKernelGGL(rest, dim3(tiles), dim3(THREADS), 0, s, M, feat, rows, logits, cdf);
}

}  // namespace sc
