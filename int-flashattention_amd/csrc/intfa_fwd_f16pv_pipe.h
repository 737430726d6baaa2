// The half-int8 and fp16/bf16 forward of intfa_fwd_f16pv.h as a software pipeline over the key blocks: head_dim 128, and head_dim 64
// in grids that leave a SIMD two waves.
//
// What bounds the kernel: a block's Q K^T, softmax and P V in turn leave the matrix pipe idle during the softmax and the vector pipe
// during the products, and with two waves per SIMD the other wave fills only part of that.  Here every MFMA of block n+1's Q K^T and of
// block n-1's P V is followed by its share of block n's softmax.  By the counters, before -> with the pipeline: fp16 B4 H32 N4096 d128
// 2.09 M -> 1.74 M clocks, matrix pipe busy 50 -> 60 % of them; half-int8 1.87 M -> 1.72 M, 42 -> 46 %.  The card lowers its clock under
// that load (1.86 -> 1.63 GHz, 1.90 -> 1.81), so the time falls by less than the clocks.  Causal half-int8 B8 H32 N2048 keeps 2.03 GHz and has neither
// pipe full (matrix 35 %, 30 % of the waves' time in waits): its workgroups are 17 key blocks long on average and fill and drain the
// pipeline each for itself, 2120 clocks per wave and block where the non-causal launch takes 1670.
// (Half-int8 with scales as lanes of a register, below: 1.65 M clocks, 48 % busy; causal 2044 clocks per wave and block, non-causal 1616.)
// B4 H32 d128, us, before -> with the pipeline: N4096 fp16 1106 -> 1038, causal 608 -> 563, half-int8 969 -> 929; N512 fp16 causal
// 27.6 -> 21.0, half-int8 30.3 -> 21.0, causal 30.1 -> 18.5.
// (Two row blocks per wave at one wave per SIMD halve the LDS reads per MFMA: fp16 N4096 another 6 %, but half-int8, whose dequantisation
// fills the issue slots, loses 15 %, and every grid of fewer than some hundred workgroups loses; not kept.)
#pragma once
#include "intfa_fwd_f16pv.h"

namespace intfa {

// QK_INT8: int8 Q/K with scales (half-int8) or 16-bit Q/K (fp16/bf16 variant).  IO_DT: type of V, P and the output
// (and of Q/K when !QK_INT8): 0 fp16, 1 bf16.
// The k_scales come as lanes of one register (scale_lane_key; us, as quads -> as lanes: B8 H32 N2048 484 -> 468, causal 299 -> 293, B4 H32 N4096 920 -> 904).
template <bool QK_INT8, int D, bool CAUSAL, int IO_DT, bool SPLIT>
__global__ void __launch_bounds__(kThreads, 2) fwd_f16pv_pipe_kernel(const KParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    static_assert(D == 64 || D == 128, "head_dim 256 runs fwd_f16pv_pair_kernel (intfa_fwd_f16pv_pair.h)");
    constexpr int BN = kBlockN16, NST = BN / 32;
    constexpr int QB = QK_INT8 ? 1 : 2;               // bytes per Q/K element
    constexpr int KROW = D * QB, VROW = D * 2;        // bytes per K row / per V row
    constexpr int KS = KROW / 32;                     // MFMA k-steps of S^T (32 bytes of a row each)
    constexpr int DT = D / 32;                        // 32-wide output tiles
    constexpr int KT = BN * KROW, VT = BN * VROW;
    constexpr int KCH = KROW / 16, VCH = VROW / 16;
    constexpr int OFF_KS = 0;
    constexpr int OFF_K = 2 * BN * 4;
    constexpr int OFF_V = OFF_K + 2 * KT;
    constexpr int LDS_BYTES = OFF_V + 2 * VT;
    __shared__ __attribute__((aligned(1024))) char smem[LDS_BYTES];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lq = lane & 31, lh = lane >> 5;

    const int n_mblk = (p.seqlen + kBlockM - 1) / kBlockM;      // the last query block may be partial
    const int n_split = SPLIT ? p.num_splits : 1;
    const WorkgroupJob wg = deal_workgroup(p, block_after_kernargs());
    const int rem = wg.rem, head = wg.b * p.heads + wg.h;
    const int mb_idx = fast_div(rem, p.d_n_split);
    const int split = rem - mb_idx * n_split;
    const int mb = CAUSAL ? n_mblk - 1 - mb_idx : mb_idx;       // heaviest query blocks first
    const int b = wg.b, h = wg.h;
    const int hk = wg.hk;                     // K/V head of this query head
    // ragged sequence lengths are handled as in the full-int8 kernel (zero-filled copies, masked last block, rows past
    // the end computed on clamped inputs and not stored)
    const int seqlen_k = keys_of_batch(p, b);
    // causal mask aligned to the bottom right corner as in the full-int8 kernel: row i sees keys 0 .. i + causal_off
    const int causal_off = seqlen_k - p.seqlen;
    const KeyBlocks kb = key_block_range<BN>(seqlen_k, CAUSAL, mb * kBlockM + kBlockM, causal_off, SPLIT, n_split, split, CAUSAL,
                                             p.blocks_per_split);
    const int nb_begin = kb.begin, nb_end = kb.end;
    const int q_row = mb * kBlockM + wave * 32 + lq;
    const bool q_valid = q_row < p.seqlen;
    const int q_ld = q_valid ? q_row : p.seqlen - 1;     // row read for lanes past the end

    // exponent scale of this lane's row: q_scale * sm_scale * log2(e) (int8 Q K^T) or sm_scale * log2(e)
    float qsc = p.qk_scale_log2;
    float m_run = -INFINITY, l_run = 0.f;
    v16f o_acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o_acc[dt][r] = 0.f;

    // ---- global -> LDS copies
    const char* Kg = p.k + b * p.k_sb + hk * p.k_sh;
    const char* Vg = p.v + b * p.v_sb + hk * p.v_sh;
    const v4i k_rsrc = make_rsrc(Kg, (uint32_t)((seqlen_k - 1) * p.k_sn + KROW));
    const v4i v_rsrc = make_rsrc(Vg, (uint32_t)((seqlen_k - 1) * p.v_sn + VROW));
    const uint32_t k_sn = (uint32_t)p.k_sn, v_sn = (uint32_t)p.v_sn;
    const auto k_lane = tile_load_lane<KROW, SWZ_K, BN>(k_sn, wave, lane);
    const auto v_lane = tile_load_lane<VROW, SWZ_V16, BN>(v_sn, wave, lane);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
    auto issue_k = [&](int nb, int buf) __attribute__((always_inline)) {
        const uint32_t off = __builtin_amdgcn_readfirstlane((nb * BN) * (int)k_sn), lds = __builtin_amdgcn_readfirstlane((int)(lds0 + OFF_K + buf * KT));
        issue_tile_load<KROW, SWZ_K, BN>(k_rsrc, off, k_sn, lds, wave, k_lane);
    };
    auto issue_v = [&](int nb, int buf) __attribute__((always_inline)) {
        const uint32_t off = __builtin_amdgcn_readfirstlane((nb * BN) * (int)v_sn), lds = __builtin_amdgcn_readfirstlane((int)(lds0 + OFF_V + buf * VT));
        issue_tile_load<VROW, SWZ_V16, BN>(v_rsrc, off, __builtin_amdgcn_readfirstlane((int)v_sn), lds, __builtin_amdgcn_readfirstlane(wave), v_lane);
    };
    // The first tiles ahead of Q and the scales, which arrive under their way from HBM (and the argument lines at once, above:
    // B16 H16 N256 half-int8 14.9 -> 13.5 us, fp16 17.2 -> 16.2, causal N2048 86.2 -> 85.7).
    // (The parity of a block counts from the end: the last one is odd.)
    const int last = nb_end - 1;
    const bool odd0 = ((nb_end - nb_begin) & 1) != 0;
    if (nb_begin < nb_end) {
        issue_k(nb_begin, odd0);
        if (nb_begin < last) issue_k(nb_begin + 1, !odd0);
    }
    // ---- Q fragments (B operand of S^T): 16 bytes per k-step
    v4i qreg[KS];
    {
        const char* qrow = p.q + b * p.q_sb + h * p.q_sh + (int64_t)q_ld * p.q_sn;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qreg[ks] = *(const v4i*)(qrow + ks * 32 + lh * 16);
    }
    const uint32_t q_scale_bits = QK_INT8 ? load_q_scale_bits(p, b, h, q_ld) : 0u;
    const KScaleSource ks_src(p, b, hk, seqlen_k);
    const bool ks_wave = wave == 0;                  // threads 0 .. 63 fetch one k_scale each (a scalar test: see fwd_full_int8_kernel)
    auto load_ks = [&](int nb) __attribute__((always_inline)) -> uint32_t {
        return (!QK_INT8 || !ks_wave) ? 0u : ks_src.load(nb * BN + tid);
    };
    const uint32_t ks_wr = OFF_KS + 4 * (tid & (BN - 1));
    auto store_ks = [&](uint32_t raw, int buf) __attribute__((always_inline)) {
        if (QK_INT8 && ks_wave) *(float*)(smem + ks_wr + buf * BN * 4) = ks_src.cvt(raw);
    };

    // ---- per-lane LDS read offsets
    const int k_swz = swz_k<KROW>(lq) & (KCH - 1);
    uint32_t k_rd[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) k_rd[ks] = OFF_K + lq * KROW + (((2 * ks + lh) ^ k_swz) << 4);
    // V through ds_read_b64_tr_b16: inside a 16-lane group, result lane i element j comes from element i%4 of the
    // 8 bytes addressed by lane 4j + i/4.  Source lane s therefore points at key row (s >> 2) of a run of four
    // consecutive keys and at the four head-dim values d0 + 4*(s & 3) .. +3, d0 = 32*dt + 16*(group & 1).
    const int g16 = lane >> 4, s16 = lane & 15;
    const int v_row0 = 4 * lh + (s16 >> 2);           // + 8*w + 16*u + 32*st
    const int v_swz = swz_v16<VROW>(v_row0) & (VCH - 1);
    uint32_t v_rd[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
        const int c = 4 * dt + 2 * (g16 & 1) + ((s16 & 3) >> 1);
        v_rd[dt] = OFF_V + v_row0 * VROW + ((c ^ v_swz) << 4) + 8 * (s16 & 1);
    }
    const uint32_t ks_rd = OFF_KS + 4 * scale_lane_key(lane);

    auto mfma16 = [&](v4i a, v4i b, v16f c) __attribute__((always_inline)) -> v16f {
        if (IO_DT == 0) return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
    };

    // ---- Software pipeline over the key blocks.  While the vector pipe evaluates the softmax of block n, the matrix pipe
    // multiplies Q K^T of block n+1 and P V of block n-1: the three are independent, and the instruction stream alternates one
    // MFMA with its share of the vector work and the LDS reads of an MFMA some places ahead.
    // (Sub-tile by sub-tile and 16 keys by 16 keys, so that a score or P fragment is dead as early as possible: the registers of
    // block n are those of block n+1.)
    // State between two blocks, by the parity of n: scores (dequantised) s, 16-bit P pf; mx: the lane's maximum over s.
    constexpr int NQ = NST * KS, NP = DT * 4;         // MFMAs of Q K^T and of P V per block
    constexpr int LA = 4;                             // an MFMA's LDS operands are requested this many MFMAs ahead
    static_assert(NST == 2, "two sub-tiles of 32 keys");
    v16f s[2][NST];
    v4i pf[2][NST][2];
    float mx = -INFINITY;

    auto k_frag = [&](int i, int kb_off) __attribute__((always_inline)) -> v4i {      // i-th MFMA of Q K^T: sub-tile i / KS, k-step i % KS
        return *(const v4i*)(smem + k_rd[i % KS] + kb_off + 32 * (i / KS) * KROW);
    };
    auto v_frag = [&](int i, int vb_off) __attribute__((always_inline)) -> v4i {      // i-th MFMA of P V: output tile i % DT, keys 16 (i / DT) ..
        const uint32_t a0 = v_rd[i % DT] + vb_off + 16 * (i / DT) * VROW;
        const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s*)INTFA_LDS(smem + a0));
        const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s*)INTFA_LDS(smem + a0 + 8 * VROW));
        return (v4i){__builtin_bit_cast(v2i, lo)[0], __builtin_bit_cast(v2i, lo)[1], __builtin_bit_cast(v2i, hi)[0], __builtin_bit_cast(v2i, hi)[1]};
    };
    // One step, PAR = n & 1: P of block n out of s[PAR] (E), Q K^T of block n+1 into s[PAR ^ 1] (QK), P V of block n-1 (PV).  The
    // first Q K^T stands alone, the last block has no next one, the last P V stands alone.  Returns the row sum of P.
    // HID: the sub-tiles of block n-1 from pv_tiles on lie past the last visible key of all the wave's rows and are not multiplied:
    // P is zero there, but zero times a V that is not finite (what a prompt's padding may hold) is not.  (A scalar test per MFMA in the
    // masked steps; half-int8 B8 H32 N2048 causal 293 -> 290 us, bf16 H32/8 N3333 190 -> 190.)
    auto step = [&](auto par_tag, auto qk_tag, auto e_tag, auto pv_tag, auto hid_tag, int pv_tiles) __attribute__((always_inline)) -> float {
        constexpr int PAR = decltype(par_tag)::value ? 1 : 0;
        constexpr bool QK = decltype(qk_tag)::value, E = decltype(e_tag)::value, PV = decltype(pv_tag)::value;
        constexpr bool HID = decltype(hid_tag)::value;
        constexpr int NQS = QK ? NQ : 0, NPS = PV ? NP : 0, NM = NQS + NPS;
        constexpr int KB = (PAR ^ 1) * KT, VB = (PAR ^ 1) * VT, SB = (PAR ^ 1) * BN * 4;
        v16i si[NST];                                  // int8 Q K^T accumulators
        v4i fr[LA];
        float ksv[NST];
        float x[32], e[32], lsum = 0.f, lfirst = 0.f;
        auto fetch = [&](int i) __attribute__((always_inline)) {
            if (i < NQS) fr[i % LA] = k_frag(i, KB);
            else if (i < NM) fr[i % LA] = v_frag(i - NQS, VB);
        };
        // element j of P: the exponent's argument two elements ahead, the exponential one ahead, then the sum and the conversion -
        // none waits for the one before it
        auto e_arg = [&](int j) __attribute__((always_inline)) { if (j < 32) { x[j] = fmaf(s[PAR][j / 16][j % 16], qsc, -m_run); asm volatile("" : "+v"(x[j])); } };
        auto e_task = [&](int j) __attribute__((always_inline)) {
            e_arg(j + 2);
            if (j + 1 < 32) { e[j + 1] = fast_exp2(x[j + 1]); asm volatile("" : "+v"(e[j + 1])); }
            // (head_dim 64: a sum per sub-tile, then their sum - the order of the decode-shaped kernel, whose waves hold a
            // sub-tile each; both give the same bits)
            if (D == 64 && j == 16) lfirst = lsum;
            lsum = j == 0 || (D == 64 && j == 16) ? e[j] : lsum + e[j];
            if (j & 1) {
                const v2f two = {e[j - 1], e[j]};
                pf[PAR][j / 16][(j % 16) / 8][(j % 8) / 2] = IO_DT == 0 ? __builtin_bit_cast(int, __builtin_convertvector(two, v2h))
                                                                      : __builtin_bit_cast(int, __builtin_convertvector(two, v2bf));
                asm volatile("" : "+v"(pf[PAR][j / 16][(j % 16) / 8][(j % 8) / 2]), "+v"(lsum));
            }
        };
        // elements 2j, 2j+1 of the next block's scores: dequantise (int8), maximum
        auto c_task = [&](int j) __attribute__((always_inline)) {
            const int st = j / 8, r = 2 * (j % 8);
            if (QK_INT8) {
#pragma unroll
                for (int k = r; k < r + 2; ++k) s[PAR ^ 1][st][k] = (float)si[st][k] * lane_scale(ksv[st], k);
            }
            mx = fmaxf(fmaxf(mx, s[PAR ^ 1][st][r]), s[PAR ^ 1][st][r + 1]);
            asm volatile("" : "+v"(mx));
        };
        auto load_kk = [&]() __attribute__((always_inline)) {
            if (QK_INT8 && QK) {
#pragma unroll
                for (int st = 0; st < NST; ++st) ksv[st] = *(const float*)(smem + ks_rd + SB + 4 * 32 * st);
            }
        };
        if (QK) mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < LA; ++i) fetch(i);
        if (E) {
            e_arg(0);
            e_arg(1);
            e[0] = fast_exp2(x[0]);
        }
        __builtin_amdgcn_sched_barrier(0);
        // vector work per MFMA: 32 elements of P over all of them, 16 pairs of scores over those of P V, two MFMAs after the last of
        // Q K^T
        constexpr int C0 = NQS + 2;
#pragma unroll
        for (int i = 0; i < NM; ++i) {
            if (i < NQS) {
                const int ks = i % KS, st = i / KS;
                if (QK_INT8) si[st] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fr[i % LA], qreg[ks], ks ? si[st] : (v16i){0}, 0, 0, 0);
                else s[PAR ^ 1][st] = mfma16(fr[i % LA], qreg[ks], ks ? s[PAR ^ 1][st] : (v16f){0});
            } else {
                const int k = i - NQS;
                if (!HID || k / DT / 2 < pv_tiles) o_acc[k % DT] = mfma16(fr[i % LA], pf[PAR ^ 1][k / DT / 2][k / DT % 2], o_acc[k % DT]);
            }
            fetch(i + LA);
            if (QK && PV && i == C0 - 4) load_kk();
            if (E) {
#pragma unroll
                for (int j = i * 32 / (NM + !NM); j < (i + 1) * 32 / (NM + !NM); ++j) e_task(j);
            }
            if (QK && PV && i >= C0) {
#pragma unroll
                for (int j = (i - C0) * 16 / (NM - C0); j < (i + 1 - C0) * 16 / (NM - C0); ++j) c_task(j);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (E && NM == 0) {
#pragma unroll
            for (int j = 0; j < 32; ++j) e_task(j);
        }
        if (QK && !PV) {
            load_kk();
#pragma unroll
            for (int j = 0; j < 16; ++j) c_task(j);
        }
        return D == 64 ? lfirst + lsum : lsum;
    };

    // sub-tiles of block nb with a key that some row of the wave sees
    auto seen_tiles = [&](int nb) __attribute__((always_inline)) -> int {
        return (mb * kBlockM + wave * 32 + 31 + causal_off - nb * BN + 32) >> 5;
    };
    // first block with a key hidden from a row: the causal diagonal's (of this query block), or the ragged last one
    const int masked_first = CAUSAL ? (mb * kBlockM + causal_off + 1) / BN : seqlen_k / BN;
    // Block nb: wait for the tiles that were requested a block ago, request those of the next step, P of the block.  MASK: the block may
    // hold hidden keys (a run-time test; the code of the plain blocks' loop has none).
    auto block = [&](auto par_tag, auto qk_tag, auto pv_tag, auto mask_tag, int nb) __attribute__((always_inline)) {
        constexpr int PAR = decltype(par_tag)::value ? 1 : 0;
        constexpr bool MASK = decltype(mask_tag)::value;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        uint32_t ks_next = 0;
        const bool more = decltype(qk_tag)::value && nb + 2 < nb_end;
        if (more) {
            issue_k(nb + 2, PAR);
            ks_next = load_ks(nb + 2);
        }
        issue_v(nb, PAR);
        const bool masked = MASK && nb >= masked_first;
        // smallest last visible key of the wave's rows, relative to the block
        const int lim_lo = (CAUSAL ? mb * kBlockM + wave * 32 + causal_off : seqlen_k - 1) - nb * BN;
        if (masked && lim_lo < BN - 1) {
            const int last = (CAUSAL ? lim_lo + lq : lim_lo) - 4 * lh;
            mx = -INFINITY;
#pragma unroll
            for (int st = 0; st < NST; ++st) {
                const uint32_t hidden = hidden_past(last - 32 * st);
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    s[PAR][st][r] = hide(s[PAR][st][r], hidden, 8 * (r >> 2) + (r & 3));
                    mx = fmaxf(mx, s[PAR][st][r]);
                }
            }
        }
        // The exponent's reference point ("frame") follows the running maximum lazily: it moves, and the output and the row
        // sum are rescaled as the reference does in every block (flash_atten_int8.py:48-52), only when some row's block
        // maximum exceeds its frame by more than kFrameSlack.  P is a 16-bit FLOATING-point number here: p' = exp2(x - frame)
        // <= 2^kFrameSlack differs from the reference's p = exp2(x - m_new) by a factor that is the same for the numerator
        // sum p' v and for the row sum, so acc / l and m + log2(l) are unchanged; only the 16-bit rounding of the single
        // p' lands on other values (relative 2^-12, unbiased).  In the common case no vector instruction touches the output.
        // (The masked blocks always move it.)  P V of the block before still adds in the old frame: the output is rescaled
        // behind it.
        const float mxs = half_pair_max(mx) * qsc;
        const bool move = masked || __builtin_amdgcn_ballot_w64(mxs > m_run + kFrameSlack) != 0;
        float a_mv = 1.f;
        if (__builtin_expect(move, 0)) {
            const float m_mv = fmaxf(m_run, mxs);
            a_mv = fast_exp2(m_run - m_mv);
            m_run = m_mv;
        }
        const float lsum = step(par_tag, qk_tag, BoolTag<true>{}, pv_tag, BoolTag<CAUSAL && MASK>{}, seen_tiles(nb - 1));
        if (__builtin_expect(move, 0)) {
#pragma clang fp contract(off)
            l_run *= a_mv;                       // (not fused with the addition below, here or in the decode-shaped kernel)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) o_acc[dt][r] *= a_mv;
        }
        {
#pragma clang fp contract(off)
            l_run += lsum;
        }
        if (QK_INT8 && decltype(qk_tag)::value) asm volatile("" : "+v"(ks_next));      // (taken for arrived on every way, also where it is not stored)
        if (more) store_ks(ks_next, PAR);
    };
    constexpr BoolTag<false> F{};
    constexpr BoolTag<true> T{};
    if (nb_begin < nb_end) {
        const uint32_t ks0 = load_ks(nb_begin), ks1 = load_ks(nb_begin < last ? nb_begin + 1 : last);
        store_ks(ks0, odd0);
        store_ks(ks1, !odd0);
        if (QK_INT8) qsc = q_scale_log2(p, q_scale_bits);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        q_has_arrived(qreg);
        __syncthreads();
        int nb = nb_begin;
        if (!odd0) {
            step(T, T, F, F, F, 0);
            block(F, T, F, T, nb++);
        } else {
            step(F, T, F, F, F, 0);
            if (nb == last) block(T, F, F, T, nb++);
            else {
                block(T, T, F, T, nb++);
                block(F, T, T, T, nb++);
            }
        }
        // plain blocks, then (causal) pairs that the diagonal crosses, then the last block
        for (; nb + 1 < last && nb + 1 < masked_first; nb += 2) {
            block(T, T, T, F, nb);
            block(F, T, T, F, nb + 1);
        }
        if (CAUSAL) {
#pragma clang loop unroll(disable)
            for (; nb < last; nb += 2) {
                block(T, T, T, T, nb);
                block(F, T, T, T, nb + 1);
            }
        }
        if (nb == last) block(T, F, T, T, nb);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        step(F, F, F, T, BoolTag<CAUSAL>{}, seen_tiles(last));
    }

    static_assert(4 * OutStage<D>::BYTES <= LDS_BYTES, "output staging fits the tile memory");
    f16pv_store<D, IO_DT, SPLIT>(smem, o_acc, m_run, l_run, nb_begin < nb_end, head, split, mb * kBlockM + wave * 32, wave, lane);
#endif  // __HIP_DEVICE_COMPILE__
}

}  // namespace intfa
