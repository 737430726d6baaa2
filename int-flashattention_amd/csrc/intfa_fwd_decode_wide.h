// Forward for few query rows per head (decoding against a key/value cache, Nq <= kDecodeMaxRows after the grouped-head fold), all three
// variants: the body of the decode-shaped kernels that intfa_fwd_decode.h and intfa_fwd_decode_f16pv.h launch for such calls.
//
// Arithmetic of the general kernels per key block (flash_atten_full_int8.py:9-71, flash_atten_int8.py:9-66, flash_atten_fp.py:9-60): S,
// dequantise, running max, P = exp2(S c - m), P requantised with the fixed scale 127 (full-int8) or cast to V's 16-bit type, P V, fp32
// accumulator scaled by alpha.
//
// What bounds a decode-shaped pass, unless it streams gigabytes, is a chain of latencies: arguments, first tiles, steps (LDS, MFMA, two
// barriers, exponentials), stores, ticket, merge.  With four waves and 32-row MFMA tiles a step of 128 keys took 1.05 us however few workgroups
// ran, most of it vector instructions on rows that do not exist.  Time line of one request against 1024 keys (full-int8 d128, 8 K/V
// heads, two splits), us from the start, before -> now: first tiles requested 1.7 -> 1.0, landed 2.9 -> 2.1, last step done 7.2 -> 4.6, ticket
// 9.2 -> 6.0, merged 11.0 -> 7.4.  So:
//   * eight waves share a step of up to 256 keys, and the MFMAs are the 16 x 16 ones: a lane holds four keys per 16-key tile of ONE of
//     16 query rows (RT = 1: up to 16 rows, four values per tile) or of two such row tiles (RT = 2: up to 32);
//   * wave w computes S^T of its NT tiles; the row maxima of the waves meet in LDS (barrier), every wave then knows the running maximum
//     of each key block of the step; it exponentiates its keys in their block's frame and publishes P (barrier); every wave multiplies
//     P of the whole step with its 16 (head_dim 256: 32) columns of V.  Head_dim 64 has four such column tiles: waves 4 - 7 take every other
//     block (16-bit V: the second half) of the step's keys, and the two sums meet in the epilogue;
//   * the first tiles are requested as soon as their addresses are known, ahead of Q, the scales and the tickets.
// The frames are those of the general full-int8 kernel: a step holds two blocks of 128 keys (head_dim 128), four of 64 (head_dim 64) or two
// of 64 (head_dim 256; one in the crowded form), and m_0 = max(m, max_0), m_1 = max(m_0, max_1), ... with the factors alpha_i = 2^(m_(i-1) - m_i).  The 16-bit P V
// variants, whose result does not depend on the frame but for the rounding of P, take one frame per step.
#pragma once
#include "intfa_device.h"
#include "intfa_launch.h"
#include "intfa_splitkv.h"
#include "intfa_fwd_f16pv.h"

namespace intfa {

constexpr int kWideWaves = 8, kWideThreads = 64 * kWideWaves;
// RT: row tiles of 16 query rows.  CROWDED (full-int8): the form with room for more workgroups per compute unit
template <int RT, bool CROWDED> struct WideRows { static constexpr int tiles = RT; static constexpr bool crowded = CROWDED; };
static_assert(kWideWaves == kMergeWaves, "");

// VI8: int8 V (full-int8); KI8: int8 Q, K
template <int D, bool KI8, bool VI8, typename R> struct WideGeom {
    static_assert(D == 64 || D == 128 || D == 256, "head dims 64, 128, 256");
    static constexpr int KROW = D * (KI8 ? 1 : 2), VROW = D * (VI8 ? 1 : 2);      // bytes per row
    // Two steps of tiles in the LDS, and room for two workgroups per compute unit where steps of at least four 16-key tiles allow it: with one, its
    // prologue and its merge (4 - 6 us) overlap with nothing.  One at head_dim 256 with 16-bit V, and for full-int8 at head_dims 128 (128 KiB of
    // tiles) and 256 in grids of at most one workgroup per unit.  Full-int8 has a second form with room for more workgroups: head_dim 128 steps of 128 keys instead of 256 (step of one request, us: 1.0 and 1.3, so the longer one while
    // there is room), head_dim 64 one step's tiles instead of two, the next ones requested once all waves hold theirs in registers
    // (three workgroups per unit instead of two, us: 640 workgroups 54 -> 39.7, 960 of 1500 keys 42.1 (128-key steps) -> 37.7), head_dim 256 steps of 64 keys,
    // whose S^T keeps half the waves busy, instead of 128 with one workgroup per unit (256 workgroups of 1500 keys 48.7 -> 41.3, 5 requests
    // of 700 11.6 -> 9.9).
    static constexpr int BUFS = VI8 && D == 64 && R::crowded ? 1 : 2;
    static constexpr int KEYS = VI8 && D < 256 && (!R::crowded || BUFS == 1) ? 256 : (D == 256 && !(VI8 && !R::crowded)) || (D == 128 && !VI8) ? 64 : 128;
    static constexpr int BNB = VI8 ? (D == 128 ? 128 : 64) : KEYS;                // keys per frame
    static constexpr int BLK = VI8 ? BNB : kBlockN16;                             // key block of the split ranges: intfa_fwd_block_n()
    static constexpr int NB = KEYS / BNB;
    // Full-int8 head_dim 256, one block per step: the row sums of even and odd blocks apart, as the form with two blocks per step has them
    static constexpr bool EVEN_ODD = VI8 && D == 256 && NB == 1;
    static constexpr int NKT = KEYS / 16;                                         // 16-key tiles per step
    static constexpr int NT = NKT >= kWideWaves ? NKT / kWideWaves : 1;           // ... per wave
    static constexpr int QKW = NKT / NT;                                          // waves with tiles of S^T
    // Tile t of wave w: w + 8 t, so that a lane adds the same keys' row sums in the same order whichever step length runs; its frame.
    __device__ static constexpr int frame_of(int w, int t) { return (w + 8 * t) / (BNB / 16); }
    static constexpr int KS = KROW / 64;                                          // MFMA k-steps of S^T
    static constexpr int TB = VI8 ? 4 : 8;                                        // bytes of P per lane and tile
    static constexpr int TPO = 16 / TB;                                           // tiles per P V MFMA
    static constexpr int NOP = NKT / TPO;                                         // P V MFMAs per step, column tile and row tile
    static constexpr int CT = D / 16;                                             // column tiles
    static constexpr int KH = CT < kWideWaves ? kWideWaves / CT : 1;              // parts of the keys that waves share
    static constexpr int CTW = CT / kWideWaves > 0 ? CT / kWideWaves : 1;         // column tiles per wave
    static constexpr int NOPW = NOP / KH;                                         // MFMAs per wave, column tile and row tile
    static constexpr int OPB = NOP / NB;                                          // ... per frame
    static_assert(!VI8 || KH == 1 || (KH == 2 && OPB == 1), "head_dim 64: waves 0 - 3 take the even blocks of a step, 4 - 7 the odd ones");
    static constexpr int KT = KEYS * KROW, VT = KEYS * VROW;
};

// Swizzles of the V tiles (see intfa_device.h): 32 lanes of a transposing read touch, 8 bytes each, the 16-byte chunk of rows 0-7 and 16-23
// (or 8-15 and 24-31) of int8 V, and two neighbouring chunks of rows 0-7 (8-15) of 16-bit V.
template <int ROW_BYTES, bool VI8> __device__ __forceinline__ int swz_v_wide(int row) {
    if (VI8) {
        if (ROW_BYTES >= 256) return (row & 7) | ((row >> 1) & 8);
        if (ROW_BYTES == 128) return ((row >> 1) & 3) | ((row >> 2) & 4);
        return ((row >> 2) & 1) | ((row >> 3) & 2);
    }
    if (ROW_BYTES >= 256) return 2 * (row & 7);
    return 2 * ((row >> 1) & 3);
}

// Copy of one tile into LDS by the eight waves: wave w issues instructions w, w + 8, ...  Both swizzles repeat within the rows that the
// eight instructions of one round cover, so a lane needs one offset.
template <int ROW_BYTES, int ROWS> struct WideTileLoad {
    static constexpr int CH = ROW_BYTES / 16, RPI = 64 / CH, NINST = ROWS * CH / 64;
    static_assert(NINST % kWideWaves == 0 && kWideWaves * RPI >= 16, "a round covers the rows that a swizzle repeats over");
    uint32_t off;
};
template <int ROW_BYTES, int ROWS, typename F>
__device__ __forceinline__ WideTileLoad<ROW_BYTES, ROWS> wide_tile_load_lane(uint32_t row_stride, int wave, int lane, F swizzle) {
    using T = WideTileLoad<ROW_BYTES, ROWS>;
    const int rsub = lane / T::CH, cp = lane % T::CH;
    return {(uint32_t)(wave * T::RPI + rsub) * row_stride + (uint32_t)((cp ^ (swizzle(wave * T::RPI + rsub) & (T::CH - 1))) << 4)};
}
// wave_lds: the wave's first 1 KiB of the tile.  (Offsets run from instruction to instruction in two scalar registers, opaque to the compiler:
// held for every instruction of both buffers they push the resources out of the scalar registers, and a step's requests took 0.4 us.)
template <bool NT, int ROW_BYTES, int ROWS>
__device__ __forceinline__ void issue_wide_tile(v4i rsrc, uint32_t tile_off, uint32_t row_stride, uint32_t wave_lds,
                                                const WideTileLoad<ROW_BYTES, ROWS>& ln) {
    using T = WideTileLoad<ROW_BYTES, ROWS>;
#pragma unroll
    for (int it = 0; it < T::NINST / kWideWaves; ++it) {
        if (it) {
            tile_off += (uint32_t)(kWideWaves * T::RPI) * row_stride;
            wave_lds += kWideWaves * 1024u;
        }
        asm volatile("" : "+s"(tile_off), "+s"(wave_lds));
        issue_copy_1k<NT>(rsrc, ln.off, tile_off, wave_lds);
    }
}

template <bool KI8> struct WideAcc { typedef v4f type; };
template <> struct WideAcc<true> { typedef v4i type; };
// IO_DT: type of the output (and of the 16-bit operands), 0 fp16, 1 bf16.  PROUND, VBLK: full-int8 only (see fwd_full_int8_kernel).
template <int D, bool KI8, bool VI8, int IO_DT, int PROUND, bool VBLK, class R>
__device__ __forceinline__ void decode_wide(const KParams& p) {
    using G = WideGeom<D, KI8, VI8, R>;
    constexpr int RT = R::tiles, ROWS = 16 * RT;
    constexpr int NB = G::NB, NT = G::NT, KS = G::KS, TB = G::TB, TPO = G::TPO, CT = G::CT, KH = G::KH, CTW = G::CTW, NOPW = G::NOPW;
    constexpr int KCH = G::KROW / 16, VCH = G::VROW / 16, BPS = G::KEYS / G::BLK;       // BPS: key blocks per step
    constexpr int NV = NB * D;                           // VBLK: channel scales per step, one row per block
    // LDS map (bytes)
    constexpr int OFF_KS = 0;                            // two fp32 k_scale vectors
    constexpr int OFF_XM = 2 * G::KEYS * 4;              // row maxima / row sums of the waves' keys, fp32
    constexpr int XW = G::NKT > kWideWaves ? G::NKT : kWideWaves;     // words per row there: one per tile; the row sums one per wave
    constexpr int OFF_XP = OFF_XM + 16 * RT * XW * 4;    // P operands: [MFMA][row tile][lane][16 bytes]
    constexpr int OFF_VS = OFF_XP + G::NOP * RT * 1024;                  // VBLK: two vectors of NV fp32 channel scales
    constexpr int OFF_K = (OFF_VS + (VBLK ? 2 * NV * 4 : 0) + 1023) / 1024 * 1024;
    constexpr int OFF_V = OFF_K + G::BUFS * G::KT;
    // (half-int8 at head_dim 128 would fit three times: a full grid of 1024 workgroups then ends with a third of the card, 247 us for 1.6 GB
    // of K and V against 234 with two)
    constexpr int LDS_BYTES = OFF_V + G::BUFS * G::VT > 56 * 1024 || D != 128 ? OFF_V + G::BUFS * G::VT : 56 * 1024;
    static_assert(LDS_BYTES <= 160 * 1024 && kMergeLds <= LDS_BYTES, "a workgroup fits the LDS of a compute unit, and the merge the workgroup's");
    static_assert(KH == 1 || CT * RT * 1024 <= G::KT, "the sums of the key parts meet in the first K tile");
    __shared__ __attribute__((aligned(1024))) char smem[LDS_BYTES];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ln = lane & 15, lh = lane >> 4;            // query row inside a row tile; which four keys of a 16-key tile

    // ---- block -> (head, block of ROWS query rows, split)
    const int n_mblk = (p.seqlen + ROWS - 1) / ROWS;
    const int n_split = p.num_splits;
    const WorkgroupJob wg = deal_workgroup(p, block_after_kernargs());
    const int mb_idx = fast_div(wg.rem, p.d_n_split), split = wg.rem - mb_idx * n_split;
    const int mb = p.causal ? n_mblk - 1 - mb_idx : mb_idx;     // heaviest query blocks first
    const int b = wg.b, h = wg.h, hk = wg.hk, group = (b * p.heads + h) * n_mblk + mb;
    const int row0 = mb * ROWS;

    const int seqlen_k = keys_of_batch(p, b);
    // causal: the row at position i sees keys 0 .. i + causal_off (bottom-right aligned); causal_rows: the rows hold several query heads of
    // one K/V group, causal_rows positions each
    const int fold = p.causal_rows;
    const int causal_off = seqlen_k - (fold ? fold : p.seqlen);
    // (a split takes blocks_per_split blocks of the whole key range, masked or not: every row of a decode-shaped problem sees nearly all keys)
    const KeyBlocks kb = key_block_range<G::BLK>(seqlen_k, p.causal != 0, fold ? fold : row0 + ROWS, causal_off, n_split > 1, n_split,
                                                 split, false, p.blocks_per_split);
    const int nb_begin = kb.begin, nb_end = kb.end;
    const int key_end = nb_end * G::BLK < seqlen_k ? nb_end * G::BLK : seqlen_k;      // one past the last key of the range

    // ---- global -> LDS copies (asynchronous, straight into LDS)
    const char* Kg = p.k + b * p.k_sb + hk * p.k_sh;
    const char* Vg = p.v + b * p.v_sb + hk * p.v_sh;
    const v4i k_rsrc = make_rsrc(Kg, (uint32_t)((seqlen_k - 1) * p.k_sn + G::KROW));
    const v4i v_rsrc = make_rsrc(Vg, (uint32_t)((seqlen_k - 1) * p.v_sn + G::VROW));
    const uint32_t k_sn = (uint32_t)p.k_sn, v_sn = (uint32_t)p.v_sn;
    const auto k_lane = wide_tile_load_lane<G::KROW, G::KEYS>(k_sn, wave, lane, [](int r) { return swz_k<G::KROW>(r); });
    const auto v_lane = wide_tile_load_lane<G::VROW, G::KEYS>(v_sn, wave, lane, [](int r) { return swz_v_wide<G::VROW, VI8>(r); });
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem + 1024u * wave;
    const bool stream = p.stream_kv != 0;
    auto issue_loads = [&](int nb, int buf) __attribute__((always_inline)) {
        const uint32_t k_off = (uint32_t)(nb * G::BLK) * k_sn, v_off = (uint32_t)(nb * G::BLK) * v_sn;
        const uint32_t k_lds = lds0 + OFF_K + buf * G::KT, v_lds = lds0 + OFF_V + buf * G::VT;
        if (stream) {
            issue_wide_tile<true>(k_rsrc, k_off, k_sn, k_lds, k_lane);
            issue_wide_tile<true>(v_rsrc, v_off, v_sn, v_lds, v_lane);
        } else {
            issue_wide_tile<false>(k_rsrc, k_off, k_sn, k_lds, k_lane);
            issue_wide_tile<false>(v_rsrc, v_off, v_sn, v_lds, v_lane);
        }
    };
    if (nb_begin < nb_end) issue_loads(nb_begin, 0);

    // ---- Q fragments (B operand of S^T = K Q^T), the same rows in every wave
    v4i qreg[RT][KS];
    uint32_t q_scale_bits[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int row = row0 + 16 * rt + ln, q_ld = row < p.seqlen ? row : p.seqlen - 1;
        const char* qrow = p.q + b * p.q_sb + h * p.q_sh + (int64_t)q_ld * p.q_sn;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qreg[rt][ks] = *(const v4i*)(qrow + ks * 64 + lh * 16);
        q_scale_bits[rt] = KI8 ? load_q_scale_bits(p, b, h, q_ld) : 0u;
    }
    const uint32_t v_scale_bits = VI8 && !VBLK ? load_scale_bits(p.v_scale, b * p.vs_sb + hk * p.vs_sh, p.scale_dtype) : 0u;
    // k_scale of a step: thread t < KEYS fetches the scale of key t; converted to fp32 when stored to LDS (whole waves: see fwd_full_int8_kernel)
    const KScaleSource ks_src(p, b, hk, seqlen_k);
    const bool ks_wave = KI8 && wave < G::KEYS / 64;
    auto load_ks = [&](int nb) __attribute__((always_inline)) -> uint32_t { return ks_src.load(nb * G::BLK + (tid & (G::KEYS - 1))); };
    const uint32_t ks_wr = OFF_KS + 4 * (tid & (G::KEYS - 1));
    // VBLK: thread NV_T0 + i fetches channel scale i of the step (block i / D, channel i % D)
    constexpr int NV_T0 = NV <= 256 ? 256 : 0;
    const bool vs_wave = VBLK && wave >= NV_T0 / 64 && wave < (NV_T0 + NV) / 64;
    const int vs_i = vs_wave ? tid - NV_T0 : 0;
    const float* Vsg = (const float*)p.v_scale + (b * p.vs_sb + hk * p.vs_sh + vs_i % D);
    // (a step's later blocks may lie past the range: their P8 are zero, and the scales of the range's last block serve - not their own, which
    // lie behind the mask and need not be finite)
    auto load_vs = [&](int nb) __attribute__((always_inline)) -> float {
        int blk = nb + vs_i / D;
        blk = blk < nb_end ? blk : nb_end - 1;
        const int row = p.vs_g == 1 ? blk : blk / p.vs_g;
        return Vsg[(int64_t)row * p.vs_sblk];
    };
    uint32_t ks_next = 0;
    float vs_next = 0.f;
    if (nb_begin < nb_end) {
        if (ks_wave) ks_next = load_ks(nb_begin);
        if (vs_wave) vs_next = load_vs(nb_begin);
    }
    const uint64_t ticket_seen = splitkv_look_at_tickets(p, group);

    float qsc[RT], m_run[RT], l_run[RT], l_odd[RT];      // l_run: this lane's keys only (EVEN_ODD: of even blocks, l_odd: of odd ones)
    v4f o_acc[CTW][RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        qsc[rt] = p.qk_scale_log2; m_run[rt] = -INFINITY; l_run[rt] = l_odd[rt] = 0.f;
#pragma unroll
        for (int j = 0; j < CTW; ++j) o_acc[j][rt] = (v4f){0.f, 0.f, 0.f, 0.f};
    }

    // ---- per-lane LDS offsets
    const int k_swz = swz_k<G::KROW>(ln) & (KCH - 1);
    uint32_t k_rd[KS];                                   // row 16 * tile + ln, chunk 4 * ks + lh
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) k_rd[ks] = OFF_K + (16 * wave + ln) * G::KROW + (((4 * ks + lh) ^ k_swz) << 4);
    // V (A operand of O^T = V^T P^T) through the transposing 8-byte loads, 16 lanes (one lh) at a time:
    //   int8:   source lane s at key row 16 * (s >> 3) + 4 * lh + ((s >> 1) & 3), 8-byte half s & 1 of the column tile's 16 bytes: two tiles a load
    //   16-bit: source lane s at key row 4 * lh + (s >> 2), 8-byte quarter s & 3 of the column tile's 32 bytes: one tile a load
    const int s16 = lane & 15;
    const int v_row = VI8 ? 16 * (s16 >> 3) + 4 * lh + ((s16 >> 1) & 3) : 4 * lh + (s16 >> 2);
    // which part of the step's keys: the odd blocks, or (16-bit V) the second half; its MFMA o is number OPS * o + kh * OPH of the step
    const int kh = KH > 1 ? wave / CT : 0;
    constexpr int OPS = VI8 ? KH : 1, OPH = VI8 ? 1 : NOPW;
    uint32_t v_rd[CTW];
#pragma unroll
    for (int j = 0; j < CTW; ++j) {
        const int ct = wave % CT + kWideWaves * j;
        const int chunk = VI8 ? ct : 2 * ct + ((s16 >> 1) & 1);
        v_rd[j] = OFF_V + (16 * TPO * OPH * kh + v_row) * G::VROW + ((chunk ^ (swz_v_wide<G::VROW, VI8>(v_row) & (VCH - 1))) << 4) + 8 * (s16 & 1);
    }
    const uint32_t kk_rd = OFF_KS + 4 * (16 * wave + 4 * lh);
    // row maxima: [row][tile]; row sums: [row][wave]
    const uint32_t xm_wr = OFF_XM + 4 * (XW * ln + wave), xm_rd = OFF_XM + 4 * XW * ln;     // + 64 * XW per row tile, + 32 per tile
    // 16-bit V and two row tiles (one key tile per wave): a lane's two rows go through the maximum together, in one exchange of lanes and one
    // store, and both rows' maxima are requested before the first is looked at.  Half-int8 d64, 32 rows of 6000 keys, us: 256 workgroups 60.3 -> 56.3, 320
    // 79.5 -> 74, 768 167 -> 160 (with all waves known to have keys, see qk_wave).  Not a quarter of the maxima per lane: fewer LDS reads, a longer chain (320: 80).
    constexpr bool TWO_ROWS = !VI8 && RT == 2;
    const uint32_t xm_wr2 = xm_wr + 64 * XW * lh;        // of row tile lh
    const uint32_t xp_wr = OFF_XP + (wave / TPO) * RT * 1024 + 16 * lane + TB * (wave % TPO);    // + 8 / TPO * RT * 1024 per tile
    const uint32_t xp_rd = OFF_XP + kh * OPH * RT * 1024 + 16 * lane;
    const uint32_t vs_wr = OFF_VS + 4 * vs_i;
    const uint32_t vs_rd = OFF_VS + 4 * (16 * (wave % CT) + 4 * lh);                  // + 4 * D per block, + 4 * 16 * kWideWaves per column tile
    const bool qk_wave = G::QKW == kWideWaves || wave < G::QKW;      // (a constant where all have: half-int8 d64 B4 H16 Nq5 Nk3001, one pass, 22.9 -> 21.0 us)
    // the smallest and the largest last visible key of the workgroup's rows, and each lane's own
    const int first_lim = p.causal ? (fold ? 0 : row0) + causal_off : 0x3fffffff;
    const int last_lim = p.causal ? (fold ? fold : row0 + ROWS) - 1 + causal_off : 0x3fffffff;
    int row_lim[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int row = row0 + 16 * rt + ln;
        row_lim[rt] = p.causal ? (fold ? row % fold : row) + causal_off : 0x3fffffff;
    }

    auto mfma_s = [&](v4i a, v4i q, auto c) __attribute__((always_inline)) {
        if constexpr (KI8) return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, q, c, 0, 0, 0);
        else if constexpr (IO_DT == 0) return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, q), c, 0, 0, 0);
        else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, q), c, 0, 0, 0);
    };
    using SAcc = typename WideAcc<KI8>::type;

    auto step = [&](auto buf_tag, int nb) __attribute__((always_inline)) {
        constexpr int BUF = decltype(buf_tag)::value ? 1 : 0;
        constexpr int KB = (G::BUFS - 1) * BUF * G::KT, VB = (G::BUFS - 1) * BUF * G::VT, SB = BUF * G::KEYS * 4, VSB = BUF * NV * 4;
        // (the scales of this step were requested right behind its tiles)
        if (ks_wave) *(float*)(smem + ks_wr + SB) = ks_src.cvt(ks_next);
        if (vs_wave) *(float*)(smem + vs_wr + VSB) = vs_next;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) q_has_arrived(qreg[rt]);
        __syncthreads();                                   // the tiles have landed; the other buffer and the exchange areas are free
        if (nb + BPS < nb_end) {
            if (G::BUFS == 2) issue_loads(nb + BPS, BUF ^ 1);
            if (ks_wave) ks_next = load_ks(nb + BPS);
            if (vs_wave) vs_next = load_vs(nb + BPS);
        }
        // -------- S^T of this wave's keys
        SAcc acc[NT][RT];
        v4f kk[NT];
        if (qk_wave) {
            v4i fr[NT][KS];
#pragma unroll
            for (int t = 0; t < NT; ++t) {
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) fr[t][ks] = *(const v4i*)(smem + k_rd[ks] + KB + 128 * t * G::KROW);
                if (KI8) kk[t] = *(const v4f*)(smem + kk_rd + SB + 512 * t);
            }
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int rt = 0; rt < RT; ++rt) acc[t][rt] = mfma_s(fr[t][ks], qreg[rt][ks], ks == 0 ? (SAcc){0, 0, 0, 0} : acc[t][rt]);
        }
        // V fragments of this wave's columns travel during the softmax
        v4i vf[CTW][NOPW];
#pragma unroll
        for (int j = 0; j < CTW; ++j)
#pragma unroll
            for (int o = 0; o < NOPW; ++o)
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const uint32_t a = v_rd[j] + VB + (16 * TPO * OPS * o + 8 * TPO * u) * G::VROW;
                    v2i x;
                    if (VI8) x = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i*)INTFA_LDS(smem + a));
                    else x = __builtin_bit_cast(v2i, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s*)INTFA_LDS(smem + a)));
                    vf[j][o][2 * u] = x[0];
                    vf[j][o][2 * u + 1] = x[1];
                }
        // -------- dequantise, row maxima of this wave's keys
        const int key0 = nb * G::BLK;
        // masked steps (wave-uniform test): keys past the end of the range, or past the first row's position
        const bool tail = key0 + G::KEYS > key_end || key0 + G::KEYS - 1 > first_lim;
        float x[NT][RT][4];
        if (qk_wave) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) x[t][rt][r] = KI8 ? (float)acc[t][rt][r] * kk[t][r] : (float)acc[t][rt][r];
            if (tail) {
                // (a branch of its own, kept one by the empty statement: folded into the loop above, the test would put a compare and a
                // select on every element of every step)
                asm volatile("");
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    const int last = (row_lim[rt] < key_end - 1 ? row_lim[rt] : key_end - 1) - key0 - 16 * wave - 4 * lh;
#pragma unroll
                    for (int t = 0; t < NT; ++t)
#pragma unroll
                        for (int r = 0; r < 4; ++r) x[t][rt][r] = hide_past(x[t][rt][r], last, 128 * t + r);
                }
            }
            if constexpr (TWO_ROWS) {
                static_assert(NT == 1, "one key tile per wave");
                float mx[RT];
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) mx[rt] = fmaxf(fmaxf(x[0][rt][0], x[0][rt][1]), fmaxf(x[0][rt][2], x[0][rt][3]));
                const float both = max_of_row_lanes(mx[0], mx[1]);
                if (lh < RT) *(float*)(smem + xm_wr2) = both;
            } else {
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    float mx[NT];
#pragma unroll
                    for (int t = 0; t < NT; ++t) mx[t] = fmaxf(fmaxf(x[t][rt][0], x[t][rt][1]), fmaxf(x[t][rt][2], x[t][rt][3]));
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        mx[t] = reduce_row_lanes(mx[t], [](float a, float c) { return fmaxf(a, c); });
                        if (lh == 0) *(float*)(smem + xm_wr + 64 * XW * rt + 32 * t) = mx[t];
                    }
                }
            }
        }
        if (G::BUFS == 1) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __syncthreads();                                   // the waves' maxima are in LDS (one buffer: its tiles are in registers)
        if (G::BUFS == 1 && nb + BPS < nb_end) issue_loads(nb + BPS, 0);
        float alpha[NB][RT], bias[RT][NT];
        float wm_all[TWO_ROWS ? RT : 1][G::NKT];
        auto read_maxima = [&](int rt) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < G::NKT / 4; ++i) *(v4f*)(wm_all[TWO_ROWS ? rt : 0] + 4 * i) = *(const v4f*)(smem + xm_rd + 64 * XW * rt + 16 * i);
        };
        if (TWO_ROWS) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) read_maxima(rt);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            if (!TWO_ROWS) read_maxima(rt);
            const float* const wm = wm_all[TWO_ROWS ? rt : 0];
            float m = m_run[rt];
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                constexpr int W = G::NKT / NB;             // tiles per frame
                float mx = wm[i * W];
#pragma unroll
                for (int w = 1; w < W; ++w) mx = fmaxf(mx, wm[i * W + w]);
                const float m_new = fmaxf(m, mx * qsc[rt]);
                alpha[i][rt] = fast_exp2(m - m_new);
                m = m_new;
                const float bi = (VI8 && PROUND == 0 ? kLog2_127 : 0.f) - m;
#pragma unroll
                for (int t = 0; t < NT; ++t) bias[rt][t] = NB == 1 || i == 0 || i == G::frame_of(wave, t) ? bi : bias[rt][t];
            }
            m_run[rt] = m;
        }
        // -------- P of this wave's keys in its block's frame; partial row sums
        if (qk_wave) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                float e[4 * NT], sum[NT];
#pragma unroll
                for (int i = 0; i < 4 * NT; ++i) {
                    e[i] = fast_exp2(fmaf(x[i / 4][rt][i % 4], qsc[rt], bias[rt][i / 4]));       // RNE mode: 127 * p
                    sum[i / 4] = i % 4 ? sum[i / 4] + e[i] : e[i];
                }
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    float own = 0.f;                       // block after block, so that the sequence does not depend on the step's length
#pragma unroll
                    for (int t = 0; t < NT; ++t) own = NB == 1 || i == G::frame_of(wave, t) ? sum[t] : own;
                    l_run[rt] = fmaf(l_run[rt], alpha[i][rt], G::EVEN_ODD && BUF ? 0.f : own);
                    if (G::EVEN_ODD) l_odd[rt] = fmaf(l_odd[rt], alpha[i][rt], BUF ? own : 0.f);
                }
                const uint32_t at = xp_wr + 1024 * rt;
                if constexpr (VI8) {
                    uint32_t pk[NT];
                    if (PROUND == 0) {
#pragma unroll
                        for (int t = 0; t < NT; ++t) {
                            pk[t] = 0;
#pragma unroll
                            for (int r = 0; r < 4; ++r) pk[t] = __builtin_amdgcn_cvt_pk_u8_f32(e[4 * t + r], r, pk[t]);
                        }
                    } else {
                        requant_p_reference<NT>(e, pk);                                   // the reference's fp16 chain
                    }
#pragma unroll
                    for (int t = 0; t < NT; ++t) *(uint32_t*)(smem + at + 8 / TPO * RT * 1024 * t) = pk[t];
                } else {
                    static_assert(VI8 || NT == 1, "16-bit P: one tile per wave");
                    if constexpr (IO_DT == 0) *(v4h*)(smem + at) = __builtin_convertvector((v4f){e[0], e[1], e[2], e[3]}, v4h);
                    else *(v4bf*)(smem + at) = __builtin_convertvector((v4f){e[0], e[1], e[2], e[3]}, v4bf);
                }
            }
        }
        v4f vsc[NB / (VI8 ? KH : 1)][CTW];                 // VBLK: channel scales of the blocks that this wave multiplies
        if (VBLK) {
#pragma unroll
            for (int i = 0; i < NB / KH; ++i)
#pragma unroll
                for (int j = 0; j < CTW; ++j) vsc[i][j] = *(const v4f*)(smem + vs_rd + VSB + 4 * D * (KH * i + kh) + 64 * kWideWaves * j);
        }
        __syncthreads();                                   // P is in LDS
        // -------- this wave's columns: O^T[d, q] = O^T alpha + V^T[d, key] P^T[key, q], block after block
        v4i pall[NOPW][RT];
#pragma unroll
        for (int o = 0; o < NOPW; ++o)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) pall[o][rt] = *(const v4i*)(smem + xp_rd + 1024 * (RT * OPS * o + rt));
        if constexpr (VI8) {
            constexpr int NBW = NB / KH;                   // blocks of this wave's keys
#pragma unroll
            for (int j = 0; j < CTW; ++j)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    v4i pv[NBW];
#pragma unroll
                    for (int i = 0; i < NBW; ++i)
#pragma unroll
                        for (int o = 0; o < G::OPB; ++o)
                            pv[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(vf[j][G::OPB * i + o], pall[G::OPB * i + o][rt], o == 0 ? (v4i){0, 0, 0, 0} : pv[i], 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        float o = o_acc[j][rt][r];
#pragma unroll
                        for (int i = 0; i < NBW; ++i) {
                            float pvf = (float)pv[i][r];
                            if (VBLK) pvf *= vsc[i][j][r];
                            if (KH == 1) o = fmaf(o, alpha[i][rt], pvf);
                            else o = fmaf(fmaf(o, alpha[KH * i][rt], kh ? 0.f : pvf), alpha[KH * i + KH - 1][rt], kh ? pvf : 0.f);
                        }
                        o_acc[j][rt][r] = o;
                    }
                }
        } else {
            if (tail) {
                // tiles past the last key that any of the rows sees: P is zero there, but zero times a V that is not finite (what a prompt's
                // padding may hold) is not
                asm volatile("");
                const int seen = (last_lim < key_end - 1 ? last_lim : key_end - 1) - key0;
#pragma unroll
                for (int o = 0; o < NOPW; ++o)
#pragma unroll
                    for (int u = 0; u < 2; ++u)
                        if (16 * (TPO * (kh * OPH + OPS * o) + u) > seen) {
#pragma unroll
                            for (int j = 0; j < CTW; ++j) vf[j][o][2 * u] = vf[j][o][2 * u + 1] = 0;
                        }
            }
#pragma unroll
            for (int j = 0; j < CTW; ++j)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) o_acc[j][rt][r] *= alpha[0][rt];
#pragma unroll
                    for (int o = 0; o < NOPW; ++o) {
                        if constexpr (IO_DT == 0) o_acc[j][rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, vf[j][o]), __builtin_bit_cast(v8h, pall[o][rt]), o_acc[j][rt], 0, 0, 0);
                        else o_acc[j][rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, vf[j][o]), __builtin_bit_cast(v8bf, pall[o][rt]), o_acc[j][rt], 0, 0, 0);
                    }
                }
        }
        // The products are consumed inside the step (int8 V), or at least not moved out of it: sunk behind the loop's branch, the first register of the
        // last one was once read without the wait states that an MFMA's result needs (the compiler counts them along the longer of two ways
        // there).  The statement emits nothing; mfma_check.py proves the distance of every reader at build time.
#pragma unroll
        for (int j = 0; j < CTW; ++j)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) asm volatile("" : "+v"(o_acc[j][rt]));
    };

    if (nb_begin < nb_end) {
        if (KI8) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) qsc[rt] = q_scale_log2(p, q_scale_bits[rt]);
        }
        int nb = nb_begin;
        while (true) {
            step(BoolTag<false>{}, nb);
            nb += BPS;
            if (nb >= nb_end) break;
            step(BoolTag<true>{}, nb);
            nb += BPS;
            if (nb >= nb_end) break;
        }
    }

    // ---- epilogue: the waves' row sums (and, at head_dim 64, the sums of the two key parts) meet in LDS; every wave scales and stores its columns
    // (the words of the row maxima and the K tiles were last read ahead of the step's last barrier)
    // (what the rest needs of the arguments is loaded again here: held since the prologue it would crowd the scalar registers of the steps;
    // all of it at once, under the exchange)
    const KernargPtr pe = kernarg_block();
    const int e_splits = pe->num_splits, e_seqlen = pe->seqlen, e_heads = pe->heads, e_batch = pe->batch, e_scale_dtype = pe->scale_dtype;
    float* const e_lse = pe->lse;
    char* const e_out = pe->out;
    const int64_t e_sb = pe->o_sb, e_sh = pe->o_sh, e_sn = pe->o_sn;
    float l_tot[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        l_tot[rt] = reduce_row_lanes(l_run[rt], [](float a, float c) { return a + c; });
        if (lh == 0 && (!G::EVEN_ODD || wave < G::QKW)) *(float*)(smem + OFF_XM + 4 * kWideWaves * (16 * rt + ln) + 4 * wave) = l_tot[rt];
        if (G::EVEN_ODD && wave < G::QKW) {
            const float odd = reduce_row_lanes(l_odd[rt], [](float a, float c) { return a + c; });
            if (lh == 0) *(float*)(smem + OFF_XM + 4 * kWideWaves * (16 * rt + ln) + 4 * (wave + G::QKW)) = odd;
        }
        if (KH > 1 && kh > 0) *(v4f*)(smem + OFF_K + 1024 * (RT * (wave % CT) + rt) + 16 * lane) = o_acc[0][rt];
    }
    asm volatile("" :: "s"(e_splits), "s"(e_seqlen), "s"(e_heads), "s"(e_batch), "s"(e_scale_dtype), "s"(e_lse), "s"(e_out), "s"(e_sb), "s"(e_sh), "s"(e_sn));
    __syncthreads();
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const v4f s0 = *(const v4f*)(smem + OFF_XM + 4 * kWideWaves * (16 * rt + ln)), s1 = *(const v4f*)(smem + OFF_XM + 4 * kWideWaves * (16 * rt + ln) + 16);
        l_tot[rt] = ((s0[0] + s0[1]) + (s0[2] + s0[3])) + ((s1[0] + s1[1]) + (s1[2] + s1[3]));
        if (KH > 1 && kh == 0) o_acc[0][rt] += *(const v4f*)(smem + OFF_K + 1024 * (RT * (wave % CT) + rt) + 16 * lane);
    }
    constexpr bool x127 = VI8 && PROUND == 0;              // the row sum is in units of 1/127
    const float vs = VI8 && !VBLK ? cvt_scale_bits(v_scale_bits, e_scale_dtype) : 1.f;
    const int rows_left = e_seqlen - row0;
    const int64_t lin0 = ((int64_t)b * e_heads + h) * e_seqlen + row0;      // the query block's first row
    auto finish = [&](auto&& put, auto&& put_lse) __attribute__((always_inline)) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            // false: an empty split range, an empty cache entry, or a causal row above the first key (zeros, lse = -inf; such a row's accumulators
            // hold NaN from exp2(-inf - -inf), hence the selects below)
            const bool seen = nb_begin < nb_end && m_run[rt] > -INFINITY;
            const float scale = !seen ? 0.f : !VI8 ? 1.f / l_tot[rt] : x127 ? vs / l_tot[rt] : vs / (127.f * l_tot[rt]);
            const int row = 16 * rt + ln;
            if (row >= rows_left) continue;
            if (KH == 1 || kh == 0) {
#pragma unroll
                for (int j = 0; j < CTW; ++j) {
                    v4f o;
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[r] = seen ? o_acc[j][rt][r] * scale : 0.f;
                    put(row, 16 * (wave % CT + kWideWaves * j) + 4 * lh, o);
                }
            }
            if (wave == 0 && lh == 0) put_lse(row, [&] { return seen ? m_run[rt] + __builtin_log2f(x127 ? l_tot[rt] * (1.f / 127.f) : l_tot[rt]) : -INFINITY; });
        }
    };
    if (e_splits > 1) {
        splitkv_open_tickets(pe, group, ticket_seen);      // (in front of this workgroup's stores: the wait for those covers it)
        const SplitPartials part(pe, D, (int64_t)split * e_batch * e_heads * e_seqlen + lin0);
        finish([&](int row, int col, v4f o) { part.put(row, D, col, o); }, [&](int row, auto&& lse) { part.put_lse(row, lse()); });
        if (pe->ticket == nullptr || !splitkv_last_arrival(pe, smem, group)) return;
        splitkv_merge_rows<D, IO_DT>(pe, smem, b, h, row0, rows_left < ROWS ? rows_left : ROWS);
    } else {
        char* const out0 = e_out + b * e_sb + h * e_sh + row0 * e_sn;
        finish([&](int row, int col, v4f o) { store_out4<IO_DT>(out0 + row * e_sn + col * 2, o); },
               [&](int row, auto&& lse) { if (e_lse != nullptr) e_lse[lin0 + row] = lse(); });
    }
}

}  // namespace intfa
