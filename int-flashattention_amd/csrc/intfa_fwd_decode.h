// Full-int8 forward whose waves share the keys: for small single-pass problems (decode_kernel_takes, intfa_capi.hip) the kernel of this file,
// for few query rows per head the one of intfa_fwd_decode_wide.h behind the same name (but at head_dim 64 with more than 16 rows
// and more workgroups than compute units: dispatch()), whose results are then the same bits.
//
// Same arithmetic as fwd_full_int8_kernel (flash_atten_full_int8.py:9-71 per 128-key block: int32 S, dequantise, running
// max, P = exp2(X c - m), P requantised with the fixed scale 127, int32 P V, fp32 accumulator), other division of labour.
// The general kernel gives each of its four waves 32 query rows; a small problem then leaves compute units without a workgroup.
// Here one workgroup owns 32 query rows and its four waves share every key block:
//   * wave w computes S^T for keys 32w .. 32w+31 of the block (KS MFMAs), dequantises and takes the partial row maxima;
//   * the partial maxima meet in LDS (barrier), every wave then holds the block's row maximum;
//   * wave w exponentiates and requantises its 32 keys and publishes its P8 fragment and row sums in LDS (barrier);
//   * wave w multiplies the whole block's P (all four fragments) with ITS 32-column slice of V and updates its slice of
//     the fp32 output.
// The int32 sums run over the same 128 keys as in the general kernel, and the waves exchange the row sums of their keys with
// the P8 fragments and add them in that kernel's order: the results are the same bits, and which of the two runs may depend on
// the number of heads and batch entries.  K/V tiles are double-buffered in LDS and the whole next tile is requested at the
// start of a block.
// Head dims 64 and 256: the general kernels' key block is 64 there (the reference admits no key block longer than head_dim,
// flash_atten_full_int8.py:88; at 256 registers set the limit), so a 128-key step of this
// kernel covers TWO blocks A (waves 0, 1) and B (waves 2, 3): after the one exchange of partial maxima every wave knows
// m_A = max(m, max_A), m_B = max(m_A, max_B) and both factors alpha_A = 2^(m - m_A), alpha_B = 2^(m_A - m_B); each wave
// requantises its keys in its own block's frame, and an output tile is updated as
// O = (O alpha_A + P8_A V_A) alpha_B + P8_B V_B with one int32 sum per block - the blocks' arithmetic of that kernel.
// FEW (head_dim 64, few query rows): the sums are those of intfa_fwd_decode_wide.h, which takes the same rows in smaller grids.  Waves 0 and 1
// multiply the A blocks with the two output tiles, waves 2 and 3 the B blocks, each into a sum of its own, and the row sums stay in the lanes, apart for each
// quad of keys, until the epilogue: the order in which that kernel's waves and lanes hold them.  Against waves 2 and 3 repeating the products of 0 and 1,
// and the row sums in the order of the general kernel, us: B16 H32/8 Nq6 Nk16000 causal 56.8 -> 53.2, B32 H16 Nq33 Nk1500 causal 34.9 -> 33.1,
// B16 H32/8 Nq5 Nk3000 16.3 -> 16.0.
#pragma once
#include "intfa_device.h"
#include "intfa_launch.h"
#include "intfa_fwd_decode_wide.h"

namespace intfa {

// Head_dim 128: one 128-key block per step, the block of the general kernel.  Head dims 64 and 256: two 64-key blocks.
template <int D, int OUT_DT /*0 f16, 1 bf16*/, int PROUND, bool VBLK, bool FEW /* few query rows: splits, grouped heads as rows, non-temporal K and V */>
__global__ void __launch_bounds__(kThreads, D <= 128 ? 2 : 1) fwd_decode_full_int8_kernel(const KParams p) {
    static_assert(D == 64 || (!FEW && (D == 128 || D == 256)), "head dims 64, 128, 256; few rows: 64");
#if defined(__HIP_DEVICE_COMPILE__)   // the host pass only needs the kernel's symbol
    constexpr int KS = D / 32;                   // k-steps of Q K^T
    constexpr int DT = D / 32;                   // 32-wide output tiles along head_dim; wave w owns tiles w, w+4, ...
    constexpr int DTW = (DT + 3) / 4;            // output tiles per wave
    constexpr int NST = 4, BN = 32 * NST;        // one 32-key sub-tile per wave
    constexpr int NSTW = FEW ? NST / 2 : NST;    // sub-tiles that a wave multiplies with V
    constexpr int NBS = D == 128 ? 1 : 2;        // key blocks (of the arithmetic) per step
    constexpr int NBW = FEW ? 1 : NBS;           // ... that a wave multiplies with V
    constexpr int BNB = BN / NBS;                // key block of the arithmetic: intfa_fwd_block_n()
    constexpr int KT = BN * D, VT = BN * D;      // bytes of one K / V tile
    constexpr int CH = D / 16;                   // 16-byte chunks per row
    constexpr int SWM = CH - 1;                  // swizzle mask of V rows
    // LDS map (bytes)
    constexpr int OFF_KS = 0;                            // two fp32 k_scale vectors
    constexpr int OFF_XM = 2 * BN * 4;                   // 4 waves x 32 rows fp32: partial row maxima
    constexpr int OFF_XP = OFF_XM + 4 * 32 * 4;          // 4 waves x 64 lanes x 16 bytes: the waves' P8 fragments
    constexpr int OFF_XS = OFF_XP + 4 * 64 * 16;         // 64 lanes x 4 waves fp32: row sums of the waves' keys
    constexpr int OFF_VS = OFF_XS + 4 * 64 * 4;          // VBLK: two vectors of NBS * D fp32 channel scales (one row per block)
    constexpr int NV = NBS * D;                          // channel scales per step
    constexpr int OFF_K = OFF_VS + (VBLK ? 2 * NV * 4 : 0);
    constexpr int OFF_V = OFF_K + 2 * KT;
    constexpr int LDS_BYTES = OFF_V + 2 * VT;
    static_assert(OFF_K % 256 == 0, "tiles keep the bank alignment the swizzles assume");
    __shared__ __attribute__((aligned(1024))) char smem[LDS_BYTES];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lq = lane & 31, lh = lane >> 5;

    // ---- block -> (head, 32-row query block, split); whole K/V heads go to one XCD as in the general kernel
    const int n_mblk = (p.seqlen + kDecodeRows - 1) / kDecodeRows;
    const WorkgroupJob wg = deal_workgroup(p, block_after_kernargs());
    const int n_split = FEW ? p.num_splits : 1;
    const int mb_idx = FEW ? fast_div(wg.rem, p.d_n_split) : wg.rem, split = wg.rem - mb_idx * n_split;
    const int mb = p.causal ? n_mblk - 1 - mb_idx : mb_idx;     // heaviest query blocks first
    const int b = wg.b, h = wg.h, hk = wg.hk, group = (b * p.heads + h) * n_mblk + mb;

    const int seqlen_k = keys_of_batch(p, b);
    // causal: row i sees keys 0 .. i + causal_off (mask aligned to the bottom right corner as in the general kernels: a few
    // new tokens against a cache); blocks past the last row's limit are not visited
    // (causal_rows: the rows hold several query heads of one K/V group, causal_rows positions each)
    const int fold = FEW ? p.causal_rows : 0;
    const int causal_off = seqlen_k - (fold ? fold : p.seqlen);
    const KeyBlocks kb = key_block_range<BNB>(seqlen_k, p.causal != 0, fold ? fold : mb * kDecodeRows + kDecodeRows, causal_off, n_split > 1,
                                              n_split, split, false, FEW ? p.blocks_per_split : 0);
    const int nb_begin = kb.begin, nb_end = kb.end;         // in blocks of BNB keys
    const int key_end = nb_end * BNB < seqlen_k ? nb_end * BNB : seqlen_k;      // one past the last key of the range
    const int q_row = mb * kDecodeRows + lq;
    const bool q_valid = q_row < p.seqlen;
    const int q_ld = q_valid ? q_row : p.seqlen - 1;

    float qsc = 0.f, m_run = -INFINITY, l_run = 0.f;
    float l_odd = 0.f;                           // head_dim 256: row sums of the odd sub-tiles (a wave of its own in that general kernel)
    float l_quad[4] = {0.f, 0.f, 0.f, 0.f};      // FEW: row sums of this lane's keys 8 a4 .. 8 a4 + 3 of every sub-tile of the wave
    float o_acc[DTW][16];
#pragma unroll
    for (int j = 0; j < DTW; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) o_acc[j][r] = 0.f;

    // ---- global -> LDS copies (asynchronous, straight into LDS; the four waves split the instructions)
    const char* Kg = p.k + b * p.k_sb + hk * p.k_sh;
    const char* Vg = p.v + b * p.v_sb + hk * p.v_sh;
    const v4i k_rsrc = make_rsrc(Kg, (uint32_t)((seqlen_k - 1) * p.k_sn + D));
    const v4i v_rsrc = make_rsrc(Vg, (uint32_t)((seqlen_k - 1) * p.v_sn + D));
    const uint32_t k_sn = (uint32_t)p.k_sn, v_sn = (uint32_t)p.v_sn;
    const auto k_lane = tile_load_lane<D, SWZ_K, BN>(k_sn, wave, lane);
    const auto v_lane = tile_load_lane<D, SWZ_V8, BN>(v_sn, wave, lane);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
    const bool stream = p.stream_kv != 0;
    auto issue_loads = [&](int nb, int buf) __attribute__((always_inline)) {
        auto issue = [&](auto nt) __attribute__((always_inline)) {
            issue_tile_load<D, SWZ_K, BN, decltype(nt)::value>(k_rsrc, (uint32_t)(nb * BNB) * k_sn, k_sn, lds0 + OFF_K + buf * KT, wave, k_lane);
            issue_tile_load<D, SWZ_V8, BN, decltype(nt)::value>(v_rsrc, (uint32_t)(nb * BNB) * v_sn, v_sn, lds0 + OFF_V + buf * VT, wave, v_lane);
        };
        if (FEW && stream) issue(BoolTag<true>{});
        else issue(BoolTag<false>{});
    };
    // The first tiles are requested ahead of everything else: Q, the scales and the lane offsets below arrive or are computed under
    // their way from HBM.
    if (nb_begin < nb_end) issue_loads(nb_begin, 0);
    uint64_t ticket_seen = 0;
    if (FEW && n_split > 1) ticket_seen = splitkv_look_at_tickets(p, group);
    // ---- Q fragment (B operand of S^T = K Q^T), the same 32 rows in every wave
    v4i qreg[KS];
    load_q8_fragments<KS>(qreg, p, b, h, q_ld, lh);
    const uint32_t q_scale_bits = load_q_scale_bits(p, b, h, q_ld);
    const uint32_t v_scale_bits = VBLK ? 0u : load_scale_bits(p.v_scale, b * p.vs_sb + hk * p.vs_sh, p.scale_dtype);
    // k_scale of a block: thread t < 128 fetches the scale of key t; converted to fp32 when stored to LDS
    const KScaleSource ks_src(p, b, hk, seqlen_k);
    auto load_ks = [&](int nb) __attribute__((always_inline)) -> uint32_t { return ks_src.load(nb * BNB + (tid & (BN - 1))); };
    auto cvt_ks = [&](uint32_t raw) __attribute__((always_inline)) -> float { return ks_src.cvt(raw); };
    // VBLK: fp32 channel scales of the step's key blocks, NV = NBS * D values.  Up to 128 values: thread 128 + i fetches
    // value i (block i / D, channel i % D); 512 values (head_dim 256): thread t fetches channel t of both blocks.
    // (per-wave tests, scalar branches: see fwd_full_int8_kernel)
    constexpr int VPT = NV > 128 ? NV / kThreads : 1;         // values per fetching thread
    const bool ks_wave = wave < BN / 64;
    const bool vs_thread = VBLK && (NV > 128 || (wave >= 2 && (wave - 2) * 64 < NV));
    const int vs_i = NV > 128 ? tid : (vs_thread ? tid - 128 : 0);
    const int vs_blk0 = NV > 128 ? 0 : vs_i / D;              // block (inside the step) of the thread's first value
    const float* Vsg = (const float*)p.v_scale + (b * p.vs_sb + hk * p.vs_sh + vs_i % D);
    // (a step's second block may lie past the range: its P8 are zero, and the scales of the range's last block serve - not its own, which
    // lie behind the mask and need not be finite)
    auto load_vs = [&](int nb, int j) __attribute__((always_inline)) -> float {
        if (!VBLK) return 0.f;
        int blk = nb + vs_blk0 + j;
        blk = blk < nb_end ? blk : nb_end - 1;
        const int row = p.vs_g == 1 ? blk : blk / p.vs_g;
        return Vsg[(int64_t)row * p.vs_sblk];
    };

    // ---- per-lane LDS offsets
    const bool blk_a = NBS == 1 || wave < 2;                          // this wave's keys belong to the first block of a step
    const int k_swz = swz_k<D>(lq) & (CH - 1);
    uint32_t k_rd[KS];                            // this wave's 32 keys: row 32*wave + lq, chunk 2*ks + lh
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) k_rd[ks] = OFF_K + (32 * wave + lq) * D + (((2 * ks + lh) ^ k_swz) << 4);
    // V through the transposing 8-byte load (see fwd_full_int8_kernel): source lane s of a 16-lane group points at key
    // row 8*(j>>2) + 4*lh + (j&3), j = s/2 (+16 for the second load, +32 per sub-tile), 8-byte half s&1
    const int g16 = lane >> 4, i16 = lane & 15, jj = i16 >> 1;
    const int v_row0 = 8 * (jj >> 2) + 4 * lh + (jj & 3);
    const int v_swz = swz_v8<D>(v_row0) & SWM;
    uint32_t v_rd[DTW];
#pragma unroll
    for (int j = 0; j < DTW; ++j) {
        const int dt = (wave + 4 * j) % DT;          // (head_dim 64: waves 2 and 3 shadow tiles 0 and 1, see below)
        const int c = 2 * dt + (g16 & 1);
        v_rd[j] = OFF_V + v_row0 * D + 8 * (i16 & 1) + (((c & SWM) ^ v_swz) << 4) + ((c & ~SWM) << 4);
        if (FEW && !blk_a) v_rd[j] += BNB * D;
    }
    const uint32_t ks_rd = OFF_KS + 4 * (32 * wave) + 16 * lh;       // + 4 * 8*a4 per read
    const uint32_t ks_wr = OFF_KS + 4 * (tid & (BN - 1));
    const uint32_t xm_wr = OFF_XM + 4 * (32 * wave + lq);
    const uint32_t xm_rd = OFF_XM + 4 * lq;                          // + 128 per wave
    const uint32_t xp_wr = OFF_XP + 1024 * wave + 16 * lane;
    const uint32_t xp_rd = OFF_XP + 16 * lane + (FEW && !blk_a ? 1024 * NSTW : 0);      // + 1024 per wave
    const uint32_t xs_rd = OFF_XS + 16 * lane, xs_wr = xs_rd + 4 * wave;
    const uint32_t vs_wr = OFF_VS + 4 * vs_i;                        // + 4 * kThreads per further value
    const uint32_t vs_rd = OFF_VS + 16 * lh + (FEW && !blk_a ? 4 * D : 0);      // + 4 * (D*blk + 32*dt + 8*a4) per read
    // head_dim 64 has two output tiles for four waves: waves 2 and 3 compute tiles 0 and 1 a second time (not FEW) and store
    // nothing (the same instruction stream for every wave; a run-time "owns a tile" test around the V fragments and the
    // accumulator update costs the owners a hundred register copies per step)
    // the last visible key of the first row of this query block, and of the lane's row
    const int first_lim = p.causal ? (fold ? 0 : mb * kDecodeRows) + causal_off : 0x3fffffff;
    const int row_lim = p.causal ? (fold ? q_row % fold : q_row) + causal_off : 0x3fffffff;

    auto step = [&](auto buf_tag, int nb) __attribute__((always_inline)) {
        constexpr int BUF = decltype(buf_tag)::value ? 1 : 0;
        constexpr int KB = BUF * KT, VB = BUF * VT, SB = BUF * BN * 4, VSB = BUF * NV * 4;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();                                   // tile nb has landed; the other buffer and the exchange areas are free
        const bool more = nb + NBS < nb_end;
        uint32_t ks_next = 0;
        float vs_next[VPT] = {};
        if (more) {
            issue_loads(nb + NBS, BUF ^ 1);
            if (ks_wave) ks_next = load_ks(nb + NBS);
            if (vs_thread) {
#pragma unroll
                for (int j = 0; j < VPT; ++j) vs_next[j] = load_vs(nb + NBS, j);
            }
        }
        // -------- S^T of this wave's 32 keys, dequantise, partial row maximum
        v4i fr[KS];
        v4f kk[4];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) fr[ks] = *(const v4i*)(smem + k_rd[ks] + KB);
#pragma unroll
        for (int a4 = 0; a4 < 4; ++a4) kk[a4] = *(const v4f*)(smem + ks_rd + SB + 4 * 8 * a4);
        v16i sacc = (v16i){0};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) sacc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fr[ks], qreg[ks], sacc, 0, 0, 0);
        // V fragments of this wave's output tiles travel during the softmax
        v4i vf[DTW][NSTW];
#pragma unroll
        for (int j = 0; j < DTW; ++j)
#pragma unroll
            for (int st = 0; st < NSTW; ++st) {
                const v2i lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                    (__attribute__((address_space(3))) v2i*)INTFA_LDS(smem + v_rd[j] + VB + (32 * st) * D));
                const v2i hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                    (__attribute__((address_space(3))) v2i*)INTFA_LDS(smem + v_rd[j] + VB + (32 * st + 16) * D));
                vf[j][st] = (v4i){lo[0], lo[1], hi[0], hi[1]};
            }
        float x[16];
        float mx = -INFINITY;
        // masked steps (wave-uniform test): keys past the end of the range (the ragged last block; with two blocks per
        // step, a second block that is not part of the range), or past the first row's position (the causal diagonal)
        const int key0 = nb * BNB;
        const bool tail = key0 + BN > key_end || key0 + BN - 1 > first_lim;
        // keys of this lane with 8*a4 + b4 >= key_lim are hidden: past the end of the range or past the lane's row
        const int last_key = (row_lim < key_end - 1 ? row_lim : key_end - 1) - key0;
        const int key_lim = last_key + 1 - 32 * wave - 4 * lh;
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = (float)sacc[r] * kk[r >> 2][r & 3];
        if (tail) {
            // (a branch of its own, kept one by the empty statement: folded into the loop above, the test would put a
            // compare and a select on every element of every step)
            asm volatile("");
#pragma unroll
            for (int r = 0; r < 16; ++r) x[r] = hide_past(x[r], key_lim - 1, 8 * (r >> 2) + (r & 3));
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, x[r]);
        mx = half_pair_max(mx);
        if (lh == 0) *(float*)(smem + xm_wr) = mx;
        __syncthreads();                                   // the four partial maxima are in LDS
        // one block per step: alpha_b = 1 and m_a = m_b is the block's maximum; two blocks: the chain A, B
        const float mx_a = fmaxf(*(const float*)(smem + xm_rd), *(const float*)(smem + xm_rd + 128));
        const float mx_b = fmaxf(*(const float*)(smem + xm_rd + 256), *(const float*)(smem + xm_rd + 384));
        const float m_a = fmaxf(m_run, (NBS == 1 ? fmaxf(mx_a, mx_b) : mx_a) * qsc);
        const float alpha = fast_exp2(m_run - m_a);
        const float m_b = NBS == 1 ? m_a : fmaxf(m_a, mx_b * qsc);
        const float alpha_b = NBS == 1 ? 1.f : fast_exp2(m_a - m_b);
        m_run = m_b;
        // -------- P of this wave's keys, requantised in its block's frame; partial row sum
        const float bias = (PROUND == 0 ? kLog2_127 : 0.f) - (blk_a ? m_a : m_b);
        float lsum = 0.f;
        v4i p8;
        {
            float e[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                e[r] = fast_exp2(fmaf(x[r], qsc, bias));                         // RNE mode: 127 * p
                if (!FEW) lsum += e[r];
            }
            if (FEW) {
#pragma unroll
                for (int a4 = 0; a4 < 4; ++a4) {
                    const float own = ((e[4 * a4] + e[4 * a4 + 1]) + e[4 * a4 + 2]) + e[4 * a4 + 3];
                    l_quad[a4] = fmaf(fmaf(l_quad[a4], alpha, blk_a ? own : 0.f), alpha_b, blk_a ? 0.f : own);
                }
            }
            if (PROUND == 0) {
#pragma unroll
                for (int w4 = 0; w4 < 4; ++w4) {
                    unsigned pk = 0;
#pragma unroll
                    for (int b4 = 0; b4 < 4; ++b4) pk = __builtin_amdgcn_cvt_pk_u8_f32(e[4 * w4 + b4], b4, pk);
                    p8[w4] = (int)pk;
                }
            } else {
                p8 = requant_p_reference16(e);                                   // the reference's fp16 chain
            }
        }
        *(v4i*)(smem + xp_wr) = p8;
        if (!FEW) *(float*)(smem + xs_wr) = lsum;
        v4f vsc[NBW][DTW][4];                              // channel scales of the step's blocks for this wave's output tiles
        if (VBLK) {
#pragma unroll
            for (int blk = 0; blk < NBW; ++blk)
#pragma unroll
                for (int j = 0; j < DTW; ++j)
#pragma unroll
                    for (int a4 = 0; a4 < 4; ++a4)
                        vsc[blk][j][a4] = *(const v4f*)(smem + vs_rd + VSB + 4 * (D * blk + 32 * ((wave + 4 * j) % DT) + 8 * a4));
        }
        __syncthreads();                                   // the four P8 fragments are in LDS
        v4i pall[NSTW];
#pragma unroll
        for (int st = 0; st < NSTW; ++st) pall[st] = *(const v4i*)(smem + xp_rd + 1024 * st);
        v4f ls = {0.f, 0.f, 0.f, 0.f};
        if (!FEW) ls = *(const v4f*)(smem + xs_rd);
        // -------- this wave's output columns: O^T[d, q] += V^T[d, key] P^T[key, q] over the whole block
#pragma unroll
        for (int j = 0; j < DTW; ++j) {
            if constexpr (FEW) {
                v16i acc = (v16i){0};
#pragma unroll
                for (int st = 0; st < NSTW; ++st) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(vf[j][st], pall[st], acc, 0, 0, 0);
                auto update = [&](auto first) __attribute__((always_inline)) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        float pv = (float)acc[r];
                        if (VBLK) pv *= vsc[0][j][r >> 2][r & 3];
                        o_acc[j][r] = fmaf(fmaf(o_acc[j][r], alpha, decltype(first)::value ? pv : 0.f), alpha_b, decltype(first)::value ? 0.f : pv);
                    }
                };
                if (blk_a) update(BoolTag<true>{});
                else update(BoolTag<false>{});
            } else if constexpr (NBS == 1) {
                v16i acc = (v16i){0};
#pragma unroll
                for (int st = 0; st < NST; ++st) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(vf[j][st], pall[st], acc, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    if (VBLK) o_acc[j][r] = fmaf(o_acc[j][r], alpha, (float)acc[r] * vsc[0][j][r >> 2][r & 3]);
                    else o_acc[j][r] = fmaf(o_acc[j][r], alpha, (float)acc[r]);
                }
            } else {
                v16i acc_a = (v16i){0}, acc_b = (v16i){0};
#pragma unroll
                for (int st = 0; st < NST / 2; ++st) acc_a = __builtin_amdgcn_mfma_i32_32x32x32_i8(vf[j][st], pall[st], acc_a, 0, 0, 0);
#pragma unroll
                for (int st = NST / 2; st < NST; ++st) acc_b = __builtin_amdgcn_mfma_i32_32x32x32_i8(vf[j][st], pall[st], acc_b, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    if (VBLK) o_acc[j][r] = fmaf(fmaf(o_acc[j][r], alpha, (float)acc_a[r] * vsc[0][j][r >> 2][r & 3]), alpha_b,
                                                 (float)acc_b[r] * vsc[NBW - 1][j][r >> 2][r & 3]);
                    else o_acc[j][r] = fmaf(fmaf(o_acc[j][r], alpha, (float)acc_a[r]), alpha_b, (float)acc_b[r]);
                }
            }
        }
        if (D == 128) l_run = fmaf(l_run, alpha, (ls[0] + ls[1]) + (ls[2] + ls[3]));
        else if (D == 64 && !FEW) l_run = fmaf(fmaf(l_run, alpha, ls[0] + ls[1]), alpha_b, ls[2] + ls[3]);
        else if (D == 256) {
            l_run = fmaf(fmaf(l_run, alpha, ls[0]), alpha_b, ls[2]);
            l_odd = fmaf(fmaf(l_odd, alpha, ls[1]), alpha_b, ls[3]);
        }
        // (the raw scale is made opaque here, behind the step's last barrier: its conversion waits for the load, and with it
        // for the next step's tile copies that were issued ahead of it - that wait belongs at the end of the step)
        asm volatile("" : "+v"(ks_next));
        if (more && ks_wave) *(float*)(smem + ks_wr + (BUF ^ 1) * BN * 4) = cvt_ks(ks_next);
        if (more && vs_thread) {
#pragma unroll
            for (int j = 0; j < VPT; ++j) *(float*)(smem + vs_wr + (BUF ^ 1) * NV * 4 + j * kThreads * 4) = vs_next[j];
        }
    };

    if (nb_begin < nb_end) {
        if (ks_wave) *(float*)(smem + ks_wr) = cvt_ks(load_ks(nb_begin));
        if (vs_thread) {
#pragma unroll
            for (int j = 0; j < VPT; ++j) *(float*)(smem + vs_wr + j * kThreads * 4) = load_vs(nb_begin, j);
        }
        qsc = q_scale_log2(p, q_scale_bits);
        int nb = nb_begin;
        while (true) {
            if (nb >= nb_end) break;
            step(BoolTag<false>{}, nb);
            nb += NBS;
            if (nb >= nb_end) break;
            step(BoolTag<true>{}, nb);
            nb += NBS;
        }
    }

    // ---- epilogue: every wave scales and stores its own output columns
    float l_tot;                                 // units of 1/127 when PROUND == 0
    if constexpr (FEW) {
        // (the words of the row maxima and the K tiles were last read ahead of the step's last barrier)
        const float t0 = half_pair_sum(l_quad[0]) + half_pair_sum(l_quad[1]), t1 = half_pair_sum(l_quad[2]) + half_pair_sum(l_quad[3]);
        static_assert(DTW == 1 && 2 * 4096 <= KT, "the sums of the two key blocks meet in the first K tile");
        if (lh == 0) *(float*)(smem + OFF_XM + 16 * lq + 4 * wave) = t0 + t1;
        if (!blk_a) {
#pragma unroll
            for (int a4 = 0; a4 < 4; ++a4)
                *(v4f*)(smem + OFF_K + 4096 * (wave - 2) + 1024 * a4 + 16 * lane) = (v4f){o_acc[0][4 * a4], o_acc[0][4 * a4 + 1], o_acc[0][4 * a4 + 2], o_acc[0][4 * a4 + 3]};
        }
        __syncthreads();
        const v4f s = *(const v4f*)(smem + OFF_XM + 16 * lq);
        l_tot = (s[0] + s[1]) + (s[2] + s[3]);
        if (blk_a) {
#pragma unroll
            for (int a4 = 0; a4 < 4; ++a4) {
                const v4f odd = *(const v4f*)(smem + OFF_K + 4096 * wave + 1024 * a4 + 16 * lane);
#pragma unroll
                for (int b4 = 0; b4 < 4; ++b4) o_acc[0][4 * a4 + b4] += odd[b4];
            }
        }
    } else {
        l_tot = half_pair_sum(l_run) + (D == 256 ? half_pair_sum(l_odd) : 0.f);
    }
    const float vs = VBLK ? 1.f : cvt_scale_bits(v_scale_bits, p.scale_dtype);
    // false: an empty split range, an empty cache entry, or a causal row above the first key (zeros, lse = -inf; such a
    // row's accumulators hold NaN from exp2(-inf - -inf), hence the selects below)
    const bool seen = nb_begin < nb_end && m_run > -INFINITY;
    const float out_scale = !seen ? 0.f : (PROUND == 0) ? (vs / l_tot) : (vs / (127.f * l_tot));
    const float l_true = (PROUND == 0) ? l_tot * (1.f / 127.f) : l_tot;
    const float lse = seen ? m_run + __builtin_log2f(l_true) : -INFINITY;
    if (FEW && n_split > 1) {
        const KernargPtr pe = kernarg_block();
        splitkv_open_tickets(pe, group, ticket_seen);
        const SplitPartials part(pe, D, ((int64_t)(split * pe->batch + b) * pe->heads + h) * pe->seqlen + mb * kDecodeRows);
        if (q_valid) {
#pragma unroll
            for (int j = 0; j < DTW; ++j) {
                const int dt = wave + 4 * j;
                if (dt >= DT) continue;
#pragma unroll
                for (int a4 = 0; a4 < 4; ++a4) {
                    v4f o;
#pragma unroll
                    for (int b4 = 0; b4 < 4; ++b4) o[b4] = seen ? o_acc[j][4 * a4 + b4] * out_scale : 0.f;
                    part.put(lq, D, 32 * dt + 8 * a4 + 4 * lh, o);
                }
            }
            if (wave == 0 && lh == 0) part.put_lse(lq, seen ? lse : -INFINITY);
        }
        if (pe->ticket == nullptr || !splitkv_last_arrival(pe, smem, group)) return;
        static_assert(kMergeLds <= LDS_BYTES, "the merge fits the tile memory");
        const int row0 = mb * kDecodeRows, rows_left = pe->seqlen - row0;
        splitkv_merge_rows<D, OUT_DT, 4>(pe, smem, b, h, row0, rows_left < kDecodeRows ? rows_left : kDecodeRows);
        return;
    }
    if (!q_valid) return;
    char* orow = p.out + b * p.o_sb + h * p.o_sh + (int64_t)q_row * p.o_sn;
#pragma unroll
    for (int j = 0; j < DTW; ++j) {
        const int dt = wave + 4 * j;
        if (dt >= DT) continue;
#pragma unroll
        for (int a4 = 0; a4 < 4; ++a4) {
            const int d0 = 32 * dt + 8 * a4 + 4 * lh;
            if (OUT_DT == 0) {
                v4h o;
#pragma unroll
                for (int b4 = 0; b4 < 4; ++b4) o[b4] = (_Float16)(seen ? o_acc[j][4 * a4 + b4] * out_scale : 0.f);
                *(v4h*)(orow + d0 * 2) = o;
            } else {
                v4s o;
#pragma unroll
                for (int b4 = 0; b4 < 4; ++b4) o[b4] = f32_to_bf16(seen ? o_acc[j][4 * a4 + b4] * out_scale : 0.f);
                *(v4s*)(orow + d0 * 2) = o;
            }
        }
    }
    if (p.lse != nullptr && wave == 0 && lh == 0) p.lse[((int64_t)b * p.heads + h) * p.seqlen + q_row] = lse;
#endif  // __HIP_DEVICE_COMPILE__
}

// Few query rows per head, split or not: intfa_fwd_decode_wide.h.
template <int D, class /* WideRows */ R, int OUT_DT, int PROUND, bool VBLK>
__global__ void __launch_bounds__(kWideThreads, (D >= 128 && !R::crowded) || (D == 256 && VBLK && R::tiles == 2) ? 2 : D == 64 && R::crowded ? 6 : 4) fwd_decode_full_int8_kernel(const KParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    decode_wide<D, true, true, OUT_DT, PROUND, VBLK, R>(p);
#endif
}

}  // namespace intfa
