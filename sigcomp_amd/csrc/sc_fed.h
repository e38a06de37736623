// sc_fed.h -- the fed decode: small and medium batches, layer 0 taken out of
// the autoregressive chain.
//
// A decode step of 32 chunks streams the 6.2 MB model through one CU (56 us
// per step, bound by the CU's 64 B/clock vector L1), and no step can start
// before the last one's symbols are known.  But of layer 0 (two thirds of
// the weights) only the window's last position needs the newest symbol; the
// other 63 are known a whole step earlier.  So the work is split by role:
//
//   * a HEAD workgroup owns 32 RT chunks.  Per step it adds the newest
//     token's position (64 KB of weights, held on chip) to layer-0 sums
//     that are already there, runs the hidden and output layers (2 MB
//     streamed per step from its XCD's L2; at RT = 1 the output layer's 128
//     KB are held in registers) and the decoder step, and publishes the
//     step's 32 RT tokens;
//   * FED_SLICES FEEDER workgroups form a set that computes those sums for up
//     to FED_SET_TILES tiles of 32 chunks.  Each feeder keeps one n-tile of
//     layer 0 (256 KB, its four waves 16 window positions each) in its
//     registers for the whole decode, so the sums of a tile cost it 64 MFMAs
//     per wave and no weight traffic; the waves' partial sums meet in LDS
//     and go to the exchange buffer.
//
// Measured per step at 2,048-token chunks: a 32-row head 20.1 us (layers 1-6
// 12.1, the last hidden layer 2.3, the output layer 1.2, the decoder step
// 2.5, layer 0's last position 1.4; 22.2 with the output layer streamed and
// the window's halves summed by the head), a 64-row head 31, a tile at its
// feeders 1.73 (1.3 of it products and operand reads, bound by the LDS: each
// operand fragment feeds one MFMA; two n-tiles over half of the window per
// feeder read half as much, 0.95, but double the sums that a head loads).
//
// While a head runs step t + 1 its feeders compute the sums of step t + 2, so
// the exchange's latency (~1.5 us each way) is off the chain, and a head's
// step is the hidden layers' L1 time (64 B/clock) plus the decoder step.
//
// Exchange of one tile (fed_bytes): two parity buffers of sums, two parity
// rows of 32 token entries, FED_SLICES * WAVES step flags.  The sums of step
// s lie in parity s & 1, written by each feeder wave with agent-coherent
// (sc1) stores and, once those have completed, announced by its flag =
// s + 1; the token of step s is the entry (s + 1) << 8 | token of parity
// s & 1 (data and flag in one word).  No buffer is overwritten while it is
// read: a feeder writes the sums of step s after it has seen the tokens of
// step s - 2, which the head publishes after it has read the sums of step
// s - 2; a head publishes the tokens of step s after it has read the sums of
// step s, for which every feeder wave had read the tokens of step s - 2.
//
// Waits are bounded (spin_max polls).  A feeder wave that times out stops
// announcing and waiting but runs its loop to the end; a head that times out
// marks its chunks SC_STATUS_SYNC_TIMEOUT and runs to its end without
// waiting, so every workgroup ends.  The launch is cooperative: all
// workgroups are resident.
#pragma once

#include "sc_kernels.h"

namespace sc {
namespace {

constexpr int FED_POS = WIN / WAVES;                 // window positions per feeder wave
constexpr int FED_KS = EDIM / 32;                    // k-steps per position

// feeder LDS: embedding table, partial sums (2 parities x 4 waves x 4 KB),
// token rings, step counts
constexpr int FED_RED_OFF = EMB_BYTES;
constexpr int FED_RED_BYTES = 2 * WAVES * 4 * 64 * 16;
constexpr int RED_READ = 5;   // position whose region reads the partial sums (a barrier before it)
constexpr int FED_TOK_OFF = FED_RED_OFF + FED_RED_BYTES;
constexpr int FED_STEPS_OFF = FED_TOK_OFF + FED_SET_TILES * WIN * 32;
constexpr int FED_FEEDER_LDS = FED_STEPS_OFF + FED_SET_TILES * 4;
static_assert(EMB_BYTES % 16 == 0, "16-byte aligned LDS parts");

// head LDS, in bytes from the start
template <int RT>
struct FedHeadLds {
    static constexpr int R = 32 * RT;
    static constexpr int EPI_N = 2;
    static constexpr int ACT = EMB_BYTES;
    static constexpr int PAR = ACT + R * PACT_ROW;
    static constexpr int SLOT = PAR + pipe_par_dwords<true>() * 4;
    static constexpr int LUT = SLOT + WAVES * EPI_N * 4 * SLOT_DWORDS * 4;
    static constexpr int LOWER = LUT + VOCAB * 8;
    static constexpr int RANGE = LOWER + R * 8;
    static constexpr int POINT = RANGE + R * 8;
    static constexpr int WOFF = POINT + R * 8;
    static constexpr int TOFF = WOFF + R * 8;
    static constexpr int RPOS = TOFF + R * 8;
    static constexpr int WCNT = RPOS + R * 4;
    static constexpr int LEN = WCNT + R * 4;
    static constexpr int STAT = LEN + R * 4;
    static constexpr int WBASE = STAT + R * 4;
    static constexpr int WBUF_OFF = WBASE + R * 4;
    static constexpr int RING = WBUF_OFF + R * WBUF * 4;
    static constexpr int LAST = RING + R * WIN;
    static constexpr int MISC = LAST + R * 2;
    // layer 0's last position, [n-tile][k-step] fragments (RES)
    static constexpr int WLAST = (MISC + 8 + 15) / 16 * 16;
    // RES: a 32-row head keeps the output layer in registers and layer 0's
    // last position in LDS; a 64-row head has neither to spare (twice the
    // accumulators and rows) and gains less: its products take as long as
    // the weight stream.
    static constexpr bool RES = RT == 1;
    static constexpr int BYTES = WLAST + (RES ? HID / 32 * FED_KS * 1024 : 0);
    static_assert(BYTES <= 160 * 1024, "LDS of a CU");
    static_assert(ACT % 16 == 0 && PAR % 16 == 0 && SLOT % 16 == 0 && LUT % 16 == 0 && MISC % 8 == 0, "alignment");
};

// LDS arrays of a head's rows
struct FedRows {
    const uint8_t *act;
    const double *lut;
    uint64_t *lower, *range, *point;
    int64_t *woff, *toff;
    int32_t *rpos, *wcnt, *len, *stat, *wbase;
    uint32_t *wbuf;
    uint8_t *ring;
    uint16_t *last;   // table address of the row's newest token
};

// Frequency step and decoder step of step t for N groups of four rows of the
// wave (rows 4 * (gi + n * WAVES) + lane / 16), as k_decompress' epilogue:
// row_freq, then the lane whose symbol's interval holds the quantile stores
// the new state (_decode_partition, cpu_entropy_coding.py:230-266).
template <int N>
__device__ __forceinline__ void fed_decode_rows(const FedRows &c, uint32_t *slots, int32_t t, int gi, int lane) {
    const int q4 = lane >> 4, u = lane & 15;
    int rr[N];
    uint64_t lower[N], range[N], point[N];
    int32_t rpos[N];
    uint32_t wnext[N];
    bool active[N];
    v4i raw[N];
#pragma unroll
    for (int n = 0; n < N; ++n) {
        const int r = (gi + n * WAVES) * 4 + q4;
        rr[n] = r;
        active[n] = t < c.len[r] && c.stat[r] == 0;
        lower[n] = c.lower[r];
        range[n] = c.range[r];
        point[n] = c.point[r];
        rpos[n] = c.rpos[r];
        // the word a renormalisation would shift in (zero past the stream's end)
        wnext[n] = c.wbuf[r * WBUF + ((rpos[n] - c.wbase[r]) & (WBUF - 1))];
        raw[n] = *(const v4i *)(c.act + pact_off(r, u));
    }
    RowFreq fr[N];
    row_freq<N>(raw, c.lut, u, fr);
    uint32_t q[N];
    bool ok[N];
#pragma unroll
    for (int n = 0; n < N; ++n) {
        const uint64_t scale = range[n] >> 24;
        q[n] = 0;
        ok[n] = scale != 0 && dec_quantile(point[n] - lower[n], scale, q[n]);
        if (ok[n] && q[n] - fr[n].ex < fr[n].tot) slot_put(slots + (n * 4 + q4) * SLOT_DWORDS, fr[n], u);
    }
    slot_sync();
#pragma unroll
    for (int n = 0; n < N; ++n) {
        const int r = rr[n];
        uint32_t cum, freq;
        const uint32_t owner = slot_get(slots + (n * 4 + q4) * SLOT_DWORDS, u, cum, freq);
        if (active[n] && ok[n] && q[n] - cum < freq) {
            const uint64_t scale = range[n] >> 24;
            uint64_t lo = lower[n] + mul_scale(scale, cum), ra = mul_scale(scale, freq), pt = point[n];
            int32_t rp = rpos[n];
            if (ra < (1ull << 32)) {
                lo <<= 32;
                ra <<= 32;
                pt = (pt << 32) | wnext[n];
                rp += 1;
            }
            c.lower[r] = lo;
            c.range[r] = ra;
            c.point[r] = pt;
            c.rpos[r] = rp;
            const int sym = (int)owner * 16 + u;
            c.ring[r * WIN + (t & (WIN - 1))] = (uint8_t)sym;
            c.last[r] = (uint16_t)emb_off(sym, 0);
        }
        if (active[n] && !ok[n] && u == 0) c.stat[r] = SC_STATUS_INVALID_STREAM;
    }
}

__device__ __forceinline__ uint32_t *fed_sync(uint8_t *xch, int tiles, int tile) {
    return (uint32_t *)(xch + (int64_t)tiles * FED_SUMS + (int64_t)tile * FED_SYNC);
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t fed_sums(uint8_t *xch, int tile, int bytes = FED_SUMS) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)(xch + (int64_t)tile * FED_SUMS), (short)0, bytes, 0x00020000);
}
// byte offset of n-tile nt's sums (4 KB: register quarter e at e * 1024 + lane * 16)
__device__ __forceinline__ int fed_sums_off(int step, int nt) { return ((step & 1) * (HID / 32) + nt) * 4096; }

// ---- feeder ------------------------------------------------------------
__device__ __forceinline__ void fed_feeder(const ModelDev &M, uint8_t *s_mem, const int32_t *__restrict__ lengths,
                                           int64_t n_chunks, int rt, int tiles, int sets, int set, int slice,
                                           uint8_t *xch, int32_t spin_max, int wave, int lane) {
    typedef unsigned v4u __attribute__((ext_vector_type(4)));
    wave = __builtin_amdgcn_readfirstlane(wave);
    const uint8_t *s_emb = s_mem;
    v4i *s_red = (v4i *)(s_mem + FED_RED_OFF);
    uint8_t *s_tok = s_mem + FED_TOK_OFF;   // [tile of the set][window slot][row]
    int32_t *s_steps = (int32_t *)(s_mem + FED_STEPS_OFF);
    const int mine = (tiles - set + sets - 1) / sets;   // tiles set, set + sets, ...
    load_emb_lds(M.emb, s_mem);
    for (int i = threadIdx.x; i < FED_SET_TILES * WIN * 32 / 4; i += THREADS) ((uint32_t *)s_tok)[i] = 0;
    if (threadIdx.x < FED_SET_TILES) s_steps[threadIdx.x] = 0;
    __syncthreads();
    // a tile's steps are its head's: the longest of the head's chunks
    for (int i = threadIdx.x; i < mine * 32 * rt; i += THREADS) {
        const int j = i / (32 * rt);
        const int64_t c = (int64_t)((set + j * sets) / rt) * (32 * rt) + i % (32 * rt);
        if (c < n_chunks) atomicMax(&s_steps[j], lengths[c]);
    }
    // this wave's weights, in registers for the whole decode: n-tile `slice`
    // over positions p0 .. p0 + 15.  The window's last position is the
    // head's: zero here, so its slot may hold any token.
    const int p0 = wave * FED_POS;
    const int g = lane >> 5, rl = lane & 31, kg = g << 4, voff = lane * 16;
    v4i w[FED_POS][FED_KS];
    v4i bias;   // of the sums this wave owns (below)
    {
        const __amdgpu_buffer_rsrc_t rs = layer_rsrc(M.layer[0]);
#pragma unroll
        for (int i = 0; i < FED_POS; ++i)
#pragma unroll
            for (int q = 0; q < FED_KS; ++q) {
                w[i][q] = wload_s(rs, voff, (slice * KT0 + (p0 + i) * FED_KS + q) * 1024);
                if (i == FED_POS - 1 && wave == WAVES - 1) w[i][q] = v4i{0, 0, 0, 0};
            }
#pragma unroll
        for (int k = 0; k < 4; ++k)   // register v of a tile: feature 8 (v / 4) + 4 g + v % 4
            bias[k] = (int)M.layer[0].par[slice * PAR_DWORDS + 8 * wave + 4 * g + k];
    }
    __syncthreads();
    const int steps_l = lane < mine ? s_steps[lane] : 0;   // lane j: steps of the set's tile j
    int maxs = 0;
    for (int j = 0; j < mine; ++j) maxs = max(maxs, __builtin_amdgcn_readlane(steps_l, j));
    // items (tile j, step s) in step order; steps past a tile's end are skipped
    auto next = [&](int &j, int &s) __attribute__((always_inline)) {
        do {
            const bool wrap = ++j >= mine;
            j = wrap ? 0 : j;
            s += wrap;
        } while (__builtin_expect(s < maxs && s >= __builtin_amdgcn_readlane(steps_l, j), 0));
        return s < maxs;
    };
    // the token entries that the sums of step s wait for
    const char *ent0 = (const char *)fed_sync(xch, tiles, set) + rl * 4;
    auto load_entries = [&](int j, int s) {
        return __hip_atomic_load((const uint32_t *)(ent0 + (uint32_t)(j * sets * FED_SYNC + (s & 1) * 128)),
                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    bool dead = false;
    // The last item's reduction: wave v sums register quarter v of the tile
    // over the four waves.  It runs beside the next item's products when
    // that item is ready, else at once (finish) before the wave polls; one
    // barrier per item either way.  s_red has two parities: a wave writes a
    // parity again only after the next item's barrier, which every reader of
    // this one has reached.
    v16i prev = {};
    bool open = false;                  // the last item's reduction is still to do
    int par = 0, poff = 0, pval = 0;    // its parity, sums offset and flag value
    int32_t *pflag = nullptr;
    int ptile = set;
    auto red_at = [&](int w_, int e) { return s_red + ((par * WAVES + w_) * 4 + e) * 64 + lane; };
    auto red_put = [&](int e) __attribute__((always_inline)) {
        *red_at(wave, e) = v4i{prev[4 * e], prev[4 * e + 1], prev[4 * e + 2], prev[4 * e + 3]};
    };
    auto announce = [&] {   // the wave's stores have completed
        wait_counts<0, 15>();
        if (lane == 0 && !dead) __hip_atomic_store(pflag, pval, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    auto finish = [&] {
        if (!open) return;
#pragma unroll
        for (int e = 0; e < 4; ++e) red_put(e);
        __syncthreads();
        v4u x = (v4u)bias;
#pragma unroll
        for (int f = 0; f < WAVES; ++f) x += (v4u)*red_at(f, wave);
        __builtin_amdgcn_raw_buffer_store_b128(x, fed_sums(xch, ptile), voff, poff, CPOL_SC1);
        announce();
        open = false;
    };
    auto tok_at = [&](int j, int s, int i) {   // slot of window position p0 + i of step s: token s - 64 + p0 + i
        return s_tok + (j * WIN + ((s + p0 + i) & (WIN - 1))) * 32 + rl;
    };
    uint32_t ent = 0;
    int j = -1, s = 0;
    bool have = next(j, s);
    int ea[FED_POS];   // the item's table addresses
#pragma unroll
    for (int i = 0; i < FED_POS; ++i) ea[i] = emb_off(SOS, 0) + kg;
    while (have) {
        // (pinned: half of the weights in accumulation registers, from which
        // an MFMA can read them, instead of copies before each use)
#pragma unroll
        for (int i = 0; i < FED_POS; ++i)
#pragma unroll
            for (int q = 0; q < FED_KS; ++q) {
                if (i >= FED_POS / 2) asm volatile("" : "+a"(w[i][q]));
                else asm volatile("" : "+v"(w[i][q]));
            }
        int jn = j, sn = s;
        const bool more = next(jn, sn);
        if (__builtin_expect(s >= 2, 1)) {
            const uint32_t want = (uint32_t)(s - 1) & 0xFFFFFFu;
            if (__builtin_expect(!dead && __builtin_amdgcn_ballot_w64((ent >> 8) != want) != 0, 0)) {
                finish();   // this item's head may be waiting for the last item
                for (int n = 0;; ++n) {
                    if (n >= spin_max) {
                        dead = true;
                        break;
                    }
                    ent = load_entries(j, s);
                    if (__builtin_amdgcn_ballot_w64((ent >> 8) != want) == 0) break;
                    __builtin_amdgcn_s_sleep(2);
                }
            }
            // every wave writes the tile's tokens (the same bytes) and reads
            // only after its own writes: no barrier
            *tok_at(j, s, WIN - 2 - p0) = (uint8_t)ent;
            // the newest token's position was not yet known when the
            // addresses were prepared
            if (p0 + FED_POS == WIN) ea[FED_POS - 2] = emb_off((int)(ent & 0xFF), 0) + kg;
        }
        // the next item's tokens travel beside this item's products
        // (unused if it is none or its step < 2)
        ent = load_entries(jn, sn);
        v4i b[2][FED_KS];
#pragma unroll
        for (int q = 0; q < FED_KS; ++q) b[0][q] = *(const v4i *)(s_emb + ea[0] + q * 32);
        v16i acc[2] = {v16i{}, v16i{}};   // two chains: one would wait for itself
        int tn[FED_POS];
        v4u part[WAVES];
        // (a reduction that finish() has done is repeated without its
        // barrier and stored nowhere: no records, and no scalar offset, which
        // the range check subtracts from their number)
        const __amdgpu_buffer_rsrc_t rs_open = fed_sums(xch, __builtin_amdgcn_readfirstlane(ptile),
                                                        __builtin_amdgcn_readfirstlane(open ? FED_SUMS : 0));
        const int off_open = __builtin_amdgcn_readfirstlane(open ? poff : 0);
        __builtin_amdgcn_sched_barrier(0);
        // One position per region: its products, the next position's operand
        // reads, the next item's address of this position, and a piece of
        // the last item's reduction.
        static_for<FED_POS>([&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value;
            if constexpr (i + 1 < FED_POS) {
#pragma unroll
                for (int q = 0; q < FED_KS; ++q) b[(i + 1) & 1][q] = *(const v4i *)(s_emb + ea[i + 1] + q * 32);
            }
            tn[i] = (int)*tok_at(jn, sn, i);
            if constexpr (i > 0) {
                ea[i - 1] = emb_off(sn + p0 + i - 1 < WIN ? SOS : tn[i - 1], 0) + kg;
                asm volatile("" : "+v"(ea[i - 1]));   // here, not after the last product
            }
            if constexpr (i < 4) red_put(i);
            if constexpr (i == RED_READ) {
#pragma unroll
                for (int f = 0; f < WAVES; ++f) part[f] = (v4u)*red_at(f, wave);
            }
            if constexpr (i == RED_READ + 1)
                __builtin_amdgcn_raw_buffer_store_b128((v4u)bias + part[0] + part[1] + part[2] + part[3], rs_open, voff,
                                                       off_open, CPOL_SC1);
#pragma unroll
            for (int q = 0; q < FED_KS; ++q)
                acc[q & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[i][q], b[i & 1][q], acc[q & 1], 0, 0, 0);
            static_for<FED_KS>([&](auto) __attribute__((always_inline)) {
                __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);   // LDS reads
                __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);   // LDS writes
                __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);   // VALU
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // MFMA
            });
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (i == RED_READ - 1) {
                if (open) __syncthreads();
            }
        });
        ea[FED_POS - 1] = emb_off(sn + p0 + FED_POS - 1 < WIN ? SOS : tn[FED_POS - 1], 0) + kg;
        if (open) announce();   // the store has had eight positions' time
        prev = acc[0] + acc[1];
        open = true;
        par ^= 1;
        poff = fed_sums_off(s, slice) + wave * 1024;
        pval = s + 1;
        ptile = set + j * sets;
        pflag = (int32_t *)fed_sync(xch, tiles, ptile) + 64 + slice * WAVES + wave;
        j = jn;
        s = sn;
        have = more;
    }
    finish();
}

// ---- head --------------------------------------------------------------

// The output layer with its weights in registers (wo[k-step][n-tile]): as
// pipe_hidden with LASTL (entry and exit conditions), without weight loads.
template <int RT>
__device__ __forceinline__ void fed_output(const LayerDev &Lp, const LayerDev &L, uint8_t *s_act, uint32_t *s_parw,
                                           int l, v16i (&accA)[PNT][RT], v16i (&accB)[PNT][RT],
                                           const v4i (&wo)[KTH][PNT], uint32_t (&pk)[PNT][RT][4], int wave, int lane) {
    constexpr int MF = PNT * RT, BLK = Slot<true>::BLK;
    const int g = lane >> 5, bbase = pact_off(lane & 31, g);
    const uint32_t *cur0 = s_parw + slot_p0(l) * BLK;
    v4i b[2][RT];
    read_b<RT>(s_act, bbase, 0, b[0]);
    const RqUni up = rq_uni(Lp);
    v16i bias[PNT];
#pragma unroll
    for (int j = 0; j < PNT; ++j) bias[j] = bias_tile<true>(cur0, j, g);
    static_for<KTH>([&](auto vc) __attribute__((always_inline)) {
        constexpr int v = decltype(vc)::value;
        if constexpr (v != 7 && v != KTH - 1) read_b<RT>(s_act, bbase, v + 1, b[(v + 1) & 1]);
        if constexpr (v < 8) rq_words_uni<true, 0, RT>(accB[v / 4], v % 4, up, pk[v / 4]);
#pragma unroll
        for (int j = 0; j < PNT; ++j)
#pragma unroll
            for (int i = 0; i < RT; ++i)
                accA[j][i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wo[v][j], b[v & 1][i], v == 0 ? bias[j] : accA[j][i],
                                                                   0, 0, 0);
        pipe_schedule<MF, (v != 7 && v != KTH - 1 ? RT : 0), 0, (v < 8 ? 12 : 0)>();
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (v == 7) {
            pstore_perm<RT>(pk, 8 + 2 * wave, s_act, lane);
            __syncthreads();
            read_b<RT>(s_act, bbase, 8, b[0]);
        }
    });
    rq_pass_uni<false, RT>(accA, rq_uni(L), pk);
    __syncthreads();
    pstore_natural<RT>(pk, 2 * wave, s_act, lane);
    __syncthreads();
}

template <int RT>
__device__ __forceinline__ void fed_head(const ModelDev &M, uint8_t *s_mem, const uint32_t *__restrict__ words,
                                         const int64_t *__restrict__ word_off, const int32_t *__restrict__ word_cnt,
                                         const int32_t *__restrict__ lengths, int64_t n_chunks,
                                         uint8_t *__restrict__ tokens, const int64_t *__restrict__ tok_off,
                                         int32_t *__restrict__ status, int tiles, int head, uint8_t *xch,
                                         int32_t spin_max, int wave, int lane) {
    using H = FedHeadLds<RT>;
    constexpr int R = H::R;
    constexpr bool UNI = true;
    wave = __builtin_amdgcn_readfirstlane(wave);
    const uint8_t *s_emb = s_mem;
    uint8_t *s_act = s_mem + H::ACT;
    uint32_t *s_par = (uint32_t *)(s_mem + H::PAR);
    uint32_t *slots = (uint32_t *)(s_mem + H::SLOT) + wave * (H::EPI_N * 4 * SLOT_DWORDS);
    int32_t *s_maxlen = (int32_t *)(s_mem + H::MISC), *s_xerr = s_maxlen + 1;
    const FedRows c{s_act,
                    (const double *)(s_mem + H::LUT),
                    (uint64_t *)(s_mem + H::LOWER),
                    (uint64_t *)(s_mem + H::RANGE),
                    (uint64_t *)(s_mem + H::POINT),
                    (int64_t *)(s_mem + H::WOFF),
                    (int64_t *)(s_mem + H::TOFF),
                    (int32_t *)(s_mem + H::RPOS),
                    (int32_t *)(s_mem + H::WCNT),
                    (int32_t *)(s_mem + H::LEN),
                    (int32_t *)(s_mem + H::STAT),
                    (int32_t *)(s_mem + H::WBASE),
                    (uint32_t *)(s_mem + H::WBUF_OFF),
                    s_mem + H::RING,
                    (uint16_t *)(s_mem + H::LAST)};
    const int64_t c0 = (int64_t)head * R;
    if (threadIdx.x == 0) {
        *s_maxlen = 0;
        *s_xerr = 0;
    }
    __syncthreads();
    for (int r = threadIdx.x; r < R; r += THREADS) {
        const int64_t ch = c0 + r;
        const bool in = ch < n_chunks;
        int32_t len = 0, cnt = 0;
        int64_t woff = 0, toff = 0;
        if (in) {
            len = lengths[ch];
            cnt = word_cnt[ch];
            woff = word_off[ch];
            toff = tok_off[ch];
        }
        int take;
        c.point[r] = dec_init_point(words + woff, cnt, take);
        c.lower[r] = 0ull;
        c.range[r] = ~0ull;
        c.rpos[r] = take;
        c.stat[r] = 0;
        c.wcnt[r] = cnt;
        c.woff[r] = woff;
        c.toff[r] = toff;
        c.len[r] = len;
        c.last[r] = (uint16_t)emb_off(SOS, 0);
        atomicMax(s_maxlen, len);
    }
    for (int i = threadIdx.x; i < R * WIN / 4; i += THREADS) ((uint32_t *)c.ring)[i] = 0;
    load_emb_lds(M.emb, s_mem);
    load_lut_lds(M.lut, (double *)(s_mem + H::LUT));
    __syncthreads();
    const int32_t steps = *s_maxlen;
    // the next 64 words of every row
    auto refill = [&] {
        for (int r = wave; r < R; r += WAVES) {
            const int32_t base = c.rpos[r], cnt = c.wcnt[r];
            c.wbuf[r * WBUF + lane] = base + lane < cnt ? words[c.woff[r] + base + lane] : 0u;
            if (lane == 0) c.wbase[r] = base;
        }
    };
    refill();
    const int voff = lane * 16, g = lane >> 5, rl = lane & 31, kg = g << 4;
    const int nb0 = 2 * wave, nb1 = 8 + 2 * wave;
    constexpr int BLK = Slot<UNI>::BLK;
    uint32_t *s_parw = s_par + wave * PIPE_SLOTS * BLK;
    constexpr int PPD = ppd<RT>();
    auto ntile = [&](int j) { return j < PNT ? nb0 + j : nb1 + j - PNT; };
    // layer 0's last window position for the wave's four n-tiles (RES: the
    // wave's own 16 KB of LDS)
    constexpr bool RES = H::RES;
    v4i *s_wlast = (v4i *)(s_mem + H::WLAST) + wave * (2 * PNT * FED_KS * 64) + lane;
    v4i wlast[RES ? 1 : 2 * PNT][FED_KS];
    {
        const __amdgpu_buffer_rsrc_t rs0 = layer_rsrc(M.layer[0]);
#pragma unroll
        for (int j = 0; j < 2 * PNT; ++j)
#pragma unroll
            for (int q = 0; q < FED_KS; ++q) {
                const v4i x = wload_s(rs0, voff, (ntile(j) * KT0 + (WIN - 1) * FED_KS + q) * 1024);
                if constexpr (RES) s_wlast[(j * FED_KS + q) * 64] = x;
                else wlast[j][q] = x;
            }
    }
    const int last = M.n_layers - 1;   // at least 3 (the launch's rule)
    v4i wo[RES ? KTH : 1][PNT];        // RES: the output layer's weights
    if constexpr (RES) {
        const __amdgpu_buffer_rsrc_t rso = layer_rsrc(M.layer[last]);
#pragma unroll
        for (int q = 0; q < KTH; ++q)
#pragma unroll
            for (int j = 0; j < PNT; ++j) wo[q][j] = wload_s(rso, voff, ((nb0 + j) * KTH + q) * 1024);
    }
    bool dead = false;
    int32_t fl[RT];   // this lane's feeder flag of each tile
#pragma unroll
    for (int i = 0; i < RT; ++i) fl[i] = -1;
    auto load_flags = [&] {
#pragma unroll
        for (int i = 0; i < RT; ++i)
            fl[i] = __hip_atomic_load((int32_t *)fed_sync(xch, tiles, head * RT + i) + 64 + lane, __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
    };
    v4i px[RT][2 * PNT][4];   // the next step's sums
    // waits for the feeders' sums of step s
    auto wait_sums = [&](int32_t s) __attribute__((always_inline)) {
        auto late = [&] {
            bool l = false;
#pragma unroll
            for (int i = 0; i < RT; ++i) l |= fl[i] <= s;
            return __builtin_amdgcn_ballot_w64(l) != 0;
        };
        if (!dead && late()) {
            for (int n = 0;; ++n) {
                if (n >= spin_max) {
                    dead = true;
                    if (lane == 0) *s_xerr = 1;
                    break;
                }
                load_flags();
                if (!late()) break;
                __builtin_amdgcn_s_sleep(2);
            }
        }
    };
    auto load_sums = [&](int32_t s) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            const __amdgpu_buffer_rsrc_t rs = fed_sums(xch, head * RT + i);
#pragma unroll
            for (int j = 0; j < 2 * PNT; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    px[i][j][e] = (v4i)__builtin_amdgcn_raw_buffer_load_b128(rs, voff, fed_sums_off(s, ntile(j)) + e * 1024,
                                                                             CPOL_SC1);
        }
    };
    const RqUni u0 = rq_uni(M.layer[0]);
    if (steps > 0) {
        wait_sums(0);
        load_sums(0);
    }
#pragma unroll 1
    for (int32_t t = 0; t < steps; ++t) {
        // (the output layer's weights stay in the accumulation registers)
        if constexpr (RES) {
#pragma unroll
            for (int q = 0; q < KTH; ++q)
#pragma unroll
                for (int j = 0; j < PNT; ++j) asm volatile("" : "+a"(wo[q][j]));
        }
        v16i accA[PNT][RT], accB[PNT][RT];
        v4i w[2][PPD][PNT];
        uint32_t pk[PNT][RT][4];
        {
            uint32_t prn[Slot<UNI>::LANE];
            par_fetch<UNI>(M.layer[1].par, nb0, lane, prn);
            const __amdgpu_buffer_rsrc_t rs1 = layer_rsrc(M.layer[1]);
#pragma unroll
            for (int x = 0; x < PPD; ++x)
#pragma unroll
                for (int j = 0; j < PNT; ++j) w[0][x][j] = wload_s(rs1, voff, ((nb0 + j) * KTH + x) * 1024);
            // layer 0: the feeders' sums plus the newest token's position
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const int ea = (int)c.last[i * 32 + rl] + kg;
                v4i b[FED_KS];
#pragma unroll
                for (int q = 0; q < FED_KS; ++q) b[q] = *(const v4i *)(s_emb + ea + q * 32);
#pragma unroll
                for (int j = 0; j < 2 * PNT; ++j) {
                    v16i &a = j < PNT ? accA[j][i] : accB[j - PNT][i];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int k = 0; k < 4; ++k) a[4 * e + k] = px[i][j][e][k];
#pragma unroll
                    for (int q = 0; q < FED_KS; ++q) {
                        v4i wl;
                        if constexpr (RES) wl = s_wlast[(j * FED_KS + q) * 64];
                        else wl = wlast[j][q];
                        a = __builtin_amdgcn_mfma_i32_32x32x32_i8(wl, b[q], a, 0, 0, 0);
                    }
                }
            }
            par_put<UNI>(s_parw + slot_p0(1) * BLK, prn, lane);
            rq_pass_uni<true, RT>(accA, u0, pk);
            pstore_perm<RT>(pk, nb0, s_act, lane);
            rq_pass_uni<true, RT>(accB, u0, pk);
            pstore_perm<RT>(pk, nb1, s_act, lane);
            __syncthreads();
        }
        pipe_hidden<RT, false, UNI, true>(M.layer[0], M.layer[1], M.layer[2], s_act, s_parw, 1, accA, accB, w, pk,
                                          wave, lane);
#pragma unroll 1
        for (int l = 2; l < last - 1; ++l)
            pipe_hidden<RT, false, UNI>(M.layer[l - 1], M.layer[l], M.layer[l + 1], s_act, s_parw, l, accA, accB, w,
                                        pk, wave, lane);
        load_flags();   // read back behind the last hidden layer
        pipe_hidden<RT, false, UNI, false, !RES>(M.layer[last - 2], M.layer[last - 1], M.layer[last], s_act,
                                                        s_parw, last - 1, accA, accB, w, pk, wave, lane);
        if constexpr (RES) {
            // the next step's sums travel beside the output layer, which
            // leaves the CU's vector L1 idle
            if (t + 1 < steps) {
                wait_sums(t + 1);
                load_sums(t + 1);
            }
            fed_output<RT>(M.layer[last - 1], M.layer[last], s_act, s_parw, last, accA, accB, wo, pk, wave, lane);
        } else {
            pipe_hidden<RT, true, UNI>(M.layer[last - 1], M.layer[last], M.layer[last], s_act, s_parw, last, accA, accB,
                                       w, pk, wave, lane);
            if (t + 1 < steps) {
                wait_sums(t + 1);
                load_sums(t + 1);
            }
        }
#pragma unroll 1
        for (int gi = wave; gi < R / 4; gi += 2 * WAVES) {
            // groups of four rows whose chunks have all ended cost nothing
            const int r0 = gi * 4 + (lane >> 4), r1 = r0 + 4 * WAVES;
            const bool a0 = __builtin_amdgcn_ballot_w64(t < c.len[r0] && c.stat[r0] == 0) != 0;
            const bool a1 = __builtin_amdgcn_ballot_w64(t < c.len[r1] && c.stat[r1] == 0) != 0;
            if (a0 && a1) fed_decode_rows<2>(c, slots, t, gi, lane);
            else if (a0) fed_decode_rows<1>(c, slots, t, gi, lane);
            else if (a1) fed_decode_rows<1>(c, slots, t, gi + WAVES, lane);
        }
        __syncthreads();
        // publish the step's tokens (rows without one repeat an old byte)
        if (t + 2 < steps && threadIdx.x < R) {
            const int r = threadIdx.x;
            __hip_atomic_store(fed_sync(xch, tiles, head * RT + r / 32) + (t & 1) * 32 + r % 32,
                               ((uint32_t)(t + 1) << 8) | c.ring[r * WIN + (t & (WIN - 1))], __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
        // every 64 steps (and at the end) the ring's tokens go out
        if ((t & (WIN - 1)) == WIN - 1 || t == steps - 1) {
            const int32_t p = (t & ~(WIN - 1)) + lane;
            for (int r = wave; r < R; r += WAVES)
                if (p <= t && p < c.len[r]) tokens[c.toff[r] + p] = c.ring[r * WIN + lane];
            refill();
        }
    }
    __syncthreads();
    for (int r = threadIdx.x; r < R; r += THREADS)
        if (c0 + r < n_chunks) status[c0 + r] = *s_xerr ? SC_STATUS_SYNC_TIMEOUT : c.stat[r];
}

// Workgroups 0 .. heads - 1 are heads, the rest feeders: set f / FED_SLICES,
// slice f % FED_SLICES.
template <int RT>
__global__ __launch_bounds__(THREADS, 1) void k_decompress_fed(ModelDev M, const uint32_t *__restrict__ words,
                                                               const int64_t *__restrict__ word_off,
                                                               const int32_t *__restrict__ word_cnt,
                                                               const int32_t *__restrict__ lengths, int64_t n_chunks,
                                                               uint8_t *__restrict__ tokens,
                                                               const int64_t *__restrict__ tok_off,
                                                               int32_t *__restrict__ status, int32_t heads,
                                                               int32_t sets, uint8_t *xch, int32_t spin_max) {
    constexpr int LDS = FedHeadLds<RT>::BYTES > FED_FEEDER_LDS ? FedHeadLds<RT>::BYTES : FED_FEEDER_LDS;
    __shared__ __attribute__((aligned(16))) uint8_t s_mem[LDS];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int tiles = heads * RT, b = (int)blockIdx.x;
    if (b < heads) {
        fed_head<RT>(M, s_mem, words, word_off, word_cnt, lengths, n_chunks, tokens, tok_off, status, tiles, b, xch,
                     spin_max, wave, lane);
    } else {
        const int f = b - heads;
        fed_feeder(M, s_mem, lengths, n_chunks, RT, tiles, sets, f / FED_SLICES, f % FED_SLICES, xch, spin_max, wave,
                   lane);
    }
}

}  // namespace
}  // namespace sc
