// Full-int8 forward at head_dim 256: eight waves per workgroup, two waves per 32 query rows.
//
// Same algorithm and the same key block (64 keys) as fwd_full_int8_kernel (flash_atten_full_int8.py:9-71), other
// division of labour.  A wave cannot hold 32 rows x 256 output columns in fp32 next to the S^T tile at two waves per
// SIMD, and giving the column halves to two independent workgroups makes both redo Q K^T and the whole softmax.  Here
// waves w and w + 4 (same SIMD) share the query rows 32w .. 32w+31:
//   * wave w + 4h computes S^T, the scaling, the row maxima, the exponentials and the int8 P of the keys 32h .. 32h+31
//     of the block (one 32-key sub-tile each);
//   * the two exchange their row maxima and their packed P fragments through LDS (the block's two workgroup barriers,
//     which also publish the V tile and the next block's K tile);
//   * wave w + 4h multiplies the whole P (64 keys) with the columns 128h .. 128h+127 of V and owns those output
//     columns; the row sum is kept per wave and added up in the epilogue.
// No vector instruction is issued twice for the same element.  Waves 0-3 copy the K tile of the next block, waves 4-7
// the V tile (both 64 rows x 256 bytes).
#pragma once
#include "intfa_device.h"

namespace intfa {

constexpr int kPairThreads = 512;

template <bool CAUSAL, int OUT_DT /*0 f16, 1 bf16*/, int PROUND, bool SPLIT, bool VBLK, bool RESIDENT>
__global__ void __launch_bounds__(kPairThreads, 1) fwd_full_int8_pair_kernel(const KParams p) {
#if defined(__HIP_DEVICE_COMPILE__)   // the host pass only needs the kernel's symbol
    constexpr int D = 256;
    constexpr int KS = D / 32;                   // k-steps of Q K^T
    constexpr int BN = 64;                       // keys per block
    constexpr int DVW = 128;                     // output columns of one wave
    constexpr int DT = DVW / 32;                 // 32-wide output tiles of one wave
    constexpr int KT = BN * D;                   // bytes of one K tile, and of one V tile
    // LDS map (bytes)
    constexpr int OFF_KS = 0;                    // two fp32 k_scale vectors
    constexpr int OFF_XM = OFF_KS + 2 * BN * 4;  // row maxima (and, in the epilogue, row sums): [wave][32]
    constexpr int OFF_VS = OFF_XM + 8 * 32 * 4;  // VBLK: two vectors of D fp32 channel scales
    constexpr int OFF_XP = OFF_VS + (VBLK ? 2 * D * 4 : 0);   // packed P fragments: [wave][lane] x 16 bytes
    constexpr int OFF_K = (OFF_XP + 8 * 64 * 16 + 1023) & ~1023;
    constexpr int OFF_V = OFF_K + 2 * KT;
    // several work items per workgroup (below): the next item's Q, and the part of the output staging that the last block's tiles have no room for
    static_assert(!RESIDENT || (!SPLIT && !VBLK), "");
    constexpr int OFF_Q = OFF_V + 2 * KT;
    constexpr int OFF_ST = OFF_Q + (RESIDENT ? kBlockM * D : 0);
    constexpr int LDS_BYTES = OFF_ST + 4 * OutStage<DVW>::BYTES;
    static_assert(2 * OutStage<DVW>::BYTES == KT && LDS_BYTES <= 160 * 1024, "output staging");
    __shared__ __attribute__((aligned(1024))) char smem[LDS_BYTES];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rw = wave & 3;                     // row group: query rows 32 rw .. 32 rw + 31 of the block
    const int hf = wave >> 2;                    // key sub-tile of the softmax work and column half of the output
    const int lq = lane & 31, lh = lane >> 5;

    // ---- work item -> (head, m-block, split), key blocks: whole K/V heads per XCD (as in fwd_full_int8_kernel)
    const int bid = block_after_kernargs();
    WorkItem it = locate_item<BN, CAUSAL, SPLIT, false>(&p, bid);
    // query row of this lane, clamped to the last one
    auto row_of = [&](auto args, const WorkItem& i) __attribute__((always_inline)) -> int {
        const int r = i.mb * kBlockM + rw * 32 + lq, n = args->seqlen;
        return r < n ? r : n - 1;
    };

    float m_run, l_run;                          // l_run: this wave's keys only
    float o_acc[DT][16];

    // ---- global -> LDS copies: waves 0-3 the K tile, waves 4-7 the V tile (same geometry, other swizzle and source)
    const uint32_t t_sn = __builtin_amdgcn_readfirstlane((uint32_t)(hf ? p.v_sn : p.k_sn));
    auto tiles_of = [&](auto args, const WorkItem& i) __attribute__((always_inline)) -> v4i {
        const char* const base = hf ? args->v + i.b * args->v_sb + i.hk * args->v_sh : args->k + i.b * args->k_sb + i.hk * args->k_sh;
        return make_rsrc(base, (uint32_t)((i.seqlen_k - 1) * (int64_t)t_sn + D));
    };
    v4i t_rsrc = tiles_of(&p, it);
    const auto k_lane = tile_load_lane<D, SWZ_K, BN>(t_sn, rw, lane);
    const auto v_lane = tile_load_lane<D, SWZ_V8, BN>(t_sn, rw, lane);
    TileLoadLane<D, SWZ_K, BN> t_lane;
    t_lane.off[0] = hf ? v_lane.off[0] : k_lane.off[0];
    static_assert(TileLoadLane<D, SWZ_K, BN>::NV == 1 && TileLoadLane<D, SWZ_V8, BN>::NV == 1, "one lane offset per tile");
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
    const uint32_t t_lds = lds0 + (hf ? OFF_V : OFF_K);
    auto issue_loads = [&](const v4i& rsrc, int nb, int buf) __attribute__((always_inline)) {
        const uint32_t off = __builtin_amdgcn_readfirstlane((nb * BN) * (int)t_sn), lds = __builtin_amdgcn_readfirstlane((int)(t_lds + buf * KT));
        issue_tile_load<D, SWZ_K, BN>(rsrc, off, t_sn, lds, rw, t_lane);
    };
    // The first item's tiles ahead of its Q, which arrives under their way from HBM (as the argument lines, at once).
    if (it.nb_begin < it.nb_end) issue_loads(t_rsrc, it.nb_begin, 0);
    // ---- Q fragment (B operand of S^T = K Q^T), resident
    v4i qreg[KS];
    load_q8_fragments<KS>(qreg, p, it.b, it.h, row_of(&p, it), lh);
    uint32_t q_scale_bits = load_q_scale_bits(p, it.b, it.h, row_of(&p, it));
    // ... of the items after the first: 128 rows through LDS
    auto issue_q = [&](const WorkItem& i) __attribute__((always_inline)) {
        const KernargPtr args = kernarg_block();
        const uint32_t q_sn = (uint32_t)args->q_sn;
        const int row0 = i.mb * kBlockM, rows = args->seqlen - row0;              // (rows past the last one: zeros)
        const v4i rsrc = make_rsrc(args->q + i.b * args->q_sb + i.h * args->q_sh + (int64_t)row0 * args->q_sn, (uint32_t)((rows < kBlockM ? rows : kBlockM) - 1) * q_sn + D);
        issue_tile_load<D, SWZ_K, kBlockM>(rsrc, 0, q_sn, lds0 + OFF_Q, rw, tile_load_lane<D, SWZ_K, kBlockM>(q_sn, rw, lane));
    };
    // k_scale of a block: thread t < 64 fetches the scale of key t; converted to fp32 when stored to LDS
    KScaleSource ks_src(&p, it.b, it.hk, it.seqlen_k);
    const int ks_key = tid & (BN - 1);
    auto load_ks = [&](int nb) __attribute__((always_inline)) -> uint32_t { return ks_src.load(nb * BN + ks_key); };   // raw bits
    auto cvt_ks = [&](uint32_t raw) __attribute__((always_inline)) -> float { return ks_src.cvt(raw); };
    // VBLK: thread 256 + c fetches the fp32 scale of channel c of the key block's scale row (vs_g key blocks per row)
    // (Which threads fetch scales is decided per WAVE, from the wave index held in a scalar register: the branches
    // below are scalar branches that leave the exec mask alone.  A per-thread test of threadIdx would mask lanes off, and
    // a register spill or reload that the compiler places in the block where such lanes rejoin runs before the mask is
    // restored there: the lanes that were off lose the value.)
    const bool ks_wave = wave == 0;              // threads 0 .. 63: one k_scale each
    const int vs_c = tid - 256;
    const bool vs_thread = VBLK && hf == 1;      // threads 256 .. 511: one channel each
    const float* Vsg = (const float*)p.v_scale + (it.b * p.vs_sb + it.hk * p.vs_sh + (vs_thread ? vs_c : 0));
    auto load_vs = [&](int nb) __attribute__((always_inline)) -> float {
        if (!VBLK) return 0.f;
        const int row = p.vs_g == 1 ? nb : nb / p.vs_g;
        return Vsg[(int64_t)row * p.vs_sblk];
    };
    const uint32_t vs_wr = OFF_VS + 4 * (vs_thread ? vs_c : 0);
    const uint32_t vs_rd = OFF_VS + 4 * DVW * hf + 16 * lh;       // + 4 * (32*dt + 8*a4) per read

    // ---- per-lane LDS read offsets
    // K (A operand of S^T): row 32 hf + lq of the tile, chunk 2 ks + lh, XOR-swizzled by the row
    // (chunk (2 ks + lh) ^ swz = (2 ks) ^ (lh ^ swz): one base per lane, k-step ks flips 32 ks in it; the tile base
    // and the row offset are multiples of 256)
    const int k_swz = swz_k<D>(lq) & 15;
    const uint32_t k_rd0 = OFF_K + (32 * hf + lq) * D + ((lh ^ k_swz) << 4);
    static_assert(OFF_K % 256 == 0 && KT % 256 == 0, "k-step XOR assumes 256-byte aligned rows");
    auto k_rd = [&](int ks) __attribute__((always_inline)) -> uint32_t { return k_rd0 ^ (uint32_t)(32 * ks); };
    // V (A operand of O^T = V^T P^T) through the transposing 8-byte load; this wave's columns start at chunk 8 hf
    const int g16 = lane >> 4, i16 = lane & 15, jj = i16 >> 1;
    const int v_row0 = 8 * (jj >> 2) + 4 * lh + (jj & 3);
    const int v_swz = swz_v8<D>(v_row0) & 15;
    uint32_t v_rd[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
        const int c = 8 * hf + 2 * dt + (g16 & 1);
        v_rd[dt] = OFF_V + v_row0 * D + 8 * (i16 & 1) + ((c ^ v_swz) << 4);
    }
    const uint32_t v_own = 32 * hf * D, v_oth = 32 * (hf ^ 1) * D;      // sub-tile of this wave's P, of the partner's
    const uint32_t ks_rd = OFF_KS + 4 * 32 * hf + 16 * lh;              // + 32 * a4 per read
    const uint32_t ks_wr = OFF_KS + 4 * (tid & (BN - 1));
    auto put_ks = [&](uint32_t raw, int buf) __attribute__((always_inline)) { *(float*)(smem + ks_wr + buf * BN * 4) = cvt_ks(raw); };
    const uint32_t xm_wr = OFF_XM + 4 * (wave * 32 + lq), xm_rd = OFF_XM + 4 * ((wave ^ 4) * 32 + lq);
    const uint32_t xp_wr = OFF_XP + 16 * (wave * 64 + lane), xp_rd = OFF_XP + 16 * ((wave ^ 4) * 64 + lane);


    // S^T accumulators of the block that is processed next (this wave's sub-tile): the MFMA chain of block nb+1 runs
    // under the accumulator update of block nb.
    v16i sacc;
    uint32_t ks_next = 0;                        // raw k_scale of the next block (threads < 64)
    float vs_pend = 0.f;                         // VBLK: channel scale of the current block, not yet in LDS (threads >= 256)

    // One key block out of LDS buffer BUF.  Keys whose index inside the block exceeds the lane's `lim` are masked (causal
    // diagonal, or the keys past the end of the sequence in its last block); the test is skipped when the wave's
    // sub-tile lies at or below the smallest `lim` of the wave.  Two workgroup barriers per block, passed by every wave:
    //   B2 publishes the row maxima (and this block's V tile and channel scales),
    //   B3 publishes the packed P (and the next block's K tile and k_scale).
    // On entry the K tile and k_scale of this block are visible and `sacc` holds this wave's S^T sub-tile.
    // In the place of a next block's tiles an item's last block requests the first ones of the item `nx`, if has_next.
    bool has_next = false, v_here = false;       // v_here: this block's V tile was awaited with the K tile
    WorkItem nx = it;
    int q_block = -1;                            // the block that requests the next item's Q
    float qsc = 0.f;
    uint32_t v_scale_bits = 0;
    // (LAST: the item's last block, one instance for both buffers.  The others have no run-time test that their place in the item would answer: the
    // two waves of a SIMD meet at the barriers, so what a scalar branch takes - some twenty of them 12 % of a block - runs under nothing.)
    auto compute = [&](auto last_tag, const int BUF, int nb) __attribute__((always_inline)) {
        constexpr bool LAST = RESIDENT && decltype(last_tag)::value, MAYBE_LAST = !RESIDENT;
        const bool more = MAYBE_LAST ? nb + 1 < it.nb_end : !LAST;
        const int VB = BUF * KT, SB = BUF * BN * 4;
        // last visible key relative to the block: smallest of the wave (uniform); the lane's, relative to its first key
        const int lim_lo = CAUSAL ? it.mb * kBlockM + rw * 32 + it.seqlen_k - p.seqlen - nb * BN : it.seqlen_k - 1 - nb * BN;
        const int lim = CAUSAL ? lim_lo + lq : lim_lo;
        int past = lim - 32 * hf - 4 * lh;
        if (RESIDENT && (CAUSAL || LAST)) asm volatile("" : "+v"(past));     // (opaque: 16 thresholds would be computed ahead of the loop)
        const bool request = more || (RESIDENT && has_next);
        const int nb_next = LAST ? nx.nb_begin : nb + 1;
        if (LAST) {
            const KernargPtr args = kernarg_block();
            if (has_next) {
                t_rsrc = tiles_of(args, nx);
                ks_src = KScaleSource(args, nx.b, nx.hk, nx.seqlen_k);
                q_scale_bits = load_scale_bits(args->q_scale, nx.b * args->qs_sb + nx.h * args->qs_sh + (int64_t)row_of(args, nx) * args->qs_sn, args->scale_dtype);
            }
            v_scale_bits = load_scale_bits(args->v_scale, it.b * args->vs_sb + it.hk * args->vs_sh, args->scale_dtype);
        }
        auto load_vfrag = [&](uint32_t sub, int dt) __attribute__((always_inline)) -> v4i {
            const v2i lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                (__attribute__((address_space(3))) v2i*)INTFA_LDS(smem + v_rd[dt] + VB + sub));
            const v2i hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                (__attribute__((address_space(3))) v2i*)INTFA_LDS(smem + v_rd[dt] + VB + sub + 16 * D));
            return (v4i){lo[0], lo[1], hi[0], hi[1]};
        };
        // the K tile of the next block goes into the other buffer (last read one block ago)
        if (request && hf == 0) {
            issue_loads(t_rsrc, nb_next, BUF ^ 1);
            ks_next = load_ks(nb_next);
        }
        // -------- pass 1: dequantise this wave's S^T sub-tile by k_scale, row maximum
        v4f kk[4];
#pragma unroll
        for (int a4 = 0; a4 < 4; ++a4) kk[a4] = *(const v4f*)(smem + ks_rd + SB + 32 * a4);
        const uint32_t hidden = RESIDENT && (CAUSAL || LAST) ? hidden_past(past) : 0u;
        float t[16];
        float mx = -INFINITY;
#pragma unroll
        for (int a4 = 0; a4 < 4; ++a4) {
            float xq[4];
#pragma unroll
            for (int b4 = 0; b4 < 4; ++b4) xq[b4] = (float)sacc[4 * a4 + b4] * kk[a4][b4];
            if ((CAUSAL || LAST || MAYBE_LAST) && 32 * hf + 31 > lim_lo) {   // wave-uniform: some lane of the wave has a hidden key here
#pragma unroll
                for (int b4 = 0; b4 < 4; ++b4) {
                    if (RESIDENT) xq[b4] = hide_number(xq[b4], hidden, 8 * a4 + b4);
                    else if (32 * hf + 8 * a4 + b4 + 4 * lh > lim) xq[b4] = -INFINITY;
                }
            }
#pragma unroll
            for (int b4 = 0; b4 < 4; ++b4) {
                t[4 * a4 + b4] = xq[b4];
                mx = fmaxf(mx, xq[b4]);
            }
        }
        mx = half_pair_max(mx);
        *(float*)(smem + xm_wr) = mx;
        if (hf == 1) {                           // this block's V tile (requested one block ago) and channel scales
            if (!RESIDENT || !v_here) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if (VBLK) *(float*)(smem + vs_wr + BUF * D * 4) = vs_pend;
        }
        __syncthreads();                         // ---- B2
        if (request && hf == 1) {                // the other V buffer was last read before this barrier
            issue_loads(t_rsrc, nb_next, BUF ^ 1);
            if (VBLK) vs_pend = load_vs(nb + 1);
            if (RESIDENT && nb == q_block) issue_q(nx);              // a block ahead of the last one (every wave has read this item's Q, and these wait next in a block's time)
        }
        mx = fmaxf(mx, *(const float*)(smem + xm_rd));
        v4i vfo[2], vfp[2];
        vfo[0] = load_vfrag(v_own, 0);
        vfp[0] = load_vfrag(v_oth, 0);
        const float m_new = fmaxf(m_run, mx * qsc);
        float alpha = fast_exp2(m_run - m_new);
        // materialised here, well ahead of the hand-written v_fma_f32 that consumes it: the result of a transcendental
        // needs a wait state before its first use, which the compiler inserts for its own instructions only
        asm volatile("" : "+v"(alpha));
        m_run = m_new;
        // -------- pass 2: P = exp2(x*qsc - m) of this wave's keys, row sum, requantise
        float lsum = 0.f;
        v4i p8o;
        const float bias = (PROUND == 0 ? kLog2_127 : 0.f) - m_new;
        if (PROUND == 0) {
#pragma unroll
            for (int w4 = 0; w4 < 4; ++w4) {
                unsigned pk = 0;
#pragma unroll
                for (int b4 = 0; b4 < 4; ++b4) {
                    const float e = fast_exp2(fmaf(t[4 * w4 + b4], qsc, bias));   // 127 * p
                    lsum += e;
                    pk = __builtin_amdgcn_cvt_pk_u8_f32(e, b4, pk);
                }
                p8o[w4] = (int)pk;
            }
        } else {
            float e[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                e[r] = fast_exp2(fmaf(t[r], qsc, bias));                          // p
                lsum += e[r];
            }
            p8o = requant_p_reference16(e);                                       // the reference's fp16 chain
        }
        *(v4i*)(smem + xp_wr) = p8o;
        // the chain of the first d-tile starts on this wave's own keys while the partner's P is on its way
        v16i oacc[2];
        oacc[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(vfo[0], p8o, (v16i){0}, 0, 0, 0);
        vfo[1] = load_vfrag(v_own, 1);
        vfp[1] = load_vfrag(v_oth, 1);
        if (more && hf == 0) {                   // the next block's K tile and k_scale
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if (ks_wave) put_ks(ks_next, BUF ^ 1);
        }
        __syncthreads();                         // ---- B3
        const v4i p8p = *(const v4i*)(smem + xp_rd);
        // K fragments of the next block (other buffer), four in flight: k-steps 2dt, 2dt+1 are consumed in stage dt and
        // their registers refilled with k-steps 2dt+4, 2dt+5
        const int KBN = (BUF ^ 1) * KT;
        v4i fr[4];
        if (more) {
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) fr[ks] = *(const v4i*)(smem + (k_rd(ks) + KBN));
        }
        oacc[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(vfp[0], p8p, oacc[0], 0, 0, 0);
        // -------- P V: O^T[d, q] += V^T[d, key] P^T[key, q]; the chain of d-tile dt+1 and a quarter of the next block's
        // Q K^T chain are issued before the accumulator update of d-tile dt
        const int VSB = BUF * D * 4;
        v4f vsc[4];
        auto load_vsc = [&](int dt) __attribute__((always_inline)) {
#pragma unroll
            for (int a4 = 0; a4 < 4; ++a4) vsc[a4] = *(const v4f*)(smem + vs_rd + VSB + 4 * (32 * dt + 8 * a4));
        };
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            __builtin_amdgcn_sched_barrier(0);
            if (VBLK) load_vsc(dt);
            if (dt + 1 < DT) {
                v16i& nacc = oacc[(dt + 1) & 1];
                nacc = __builtin_amdgcn_mfma_i32_32x32x32_i8(vfo[(dt + 1) & 1], p8o, (v16i){0}, 0, 0, 0);
                nacc = __builtin_amdgcn_mfma_i32_32x32x32_i8(vfp[(dt + 1) & 1], p8p, nacc, 0, 0, 0);
            }
            if (more) {
#pragma unroll
                for (int ks = 2 * dt; ks < 2 * dt + 2; ++ks) {
                    if (ks == 0) sacc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fr[0], qreg[0], (v16i){0}, 0, 0, 0);
                    else sacc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fr[ks & 3], qreg[ks], sacc, 0, 0, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            if (more && 2 * dt + 4 < KS) {
#pragma unroll
                for (int ks = 2 * dt + 4; ks < 2 * dt + 6; ++ks) fr[ks & 3] = *(const v4i*)(smem + (k_rd(ks) + KBN));
            }
            if (dt + 2 < DT) {                   // fragments of d-tile dt+2 replace those of dt, whose chain has been issued
                vfo[dt & 1] = load_vfrag(v_own, dt + 2);
                vfp[dt & 1] = load_vfrag(v_oth, dt + 2);
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                float pv = (float)oacc[dt & 1][r];
                if (VBLK) pv *= vsc[r >> 2][r & 3];
                asm volatile("v_fma_f32 %0, %0, %1, %2" : "+v"(o_acc[dt][r]) : "v"(alpha), "v"(pv));
            }
        }
        l_run = fmaf(l_run, alpha, lsum);
    };

    // ---- Work items of this workgroup.  One while all of the launch's workgroups are resident; with more items (RESIDENT) one workgroup per compute
    // unit takes every grid-th, in the order in which the hardware would deal them (causal: every second round backwards, so that the sums of
    // the lengths agree).  What it is for: a workgroup fills its compute unit, and nothing ran under its first loads and its last stores (20 % of the time
    // at 1024 keys).  So an item's last block requests the next one's first tiles and the block before it Q (into the LDS), and the stores have until
    // the next item's first wait for tiles, a part of a key block (waves 4-7: one more block; an item of one block: its end).  us, one item
    // per workgroup -> this: B16 H16 N1024 bf16 255 -> 238, causal 169 -> 155, B4 H32 N2048 448 -> 422, B32 H32 N128 causal 43.7 -> 37.6; what
    // bounds it then is the loop over the key blocks.  Launches of one round lose 5 % in the longer code: they run the other form.
    int buf = 0;                                 // LDS buffer of the item's first block, then of its last
    int round = 0;
    if (it.nb_begin < it.nb_end) {
        const uint32_t s0 = load_ks(it.nb_begin);
        if (ks_wave) put_ks(s0, 0);
        if (vs_thread) vs_pend = load_vs(it.nb_begin);
        qsc = q_scale_log2(p, q_scale_bits);
        if (hf == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }
    q_has_arrived(qreg);                         // (outside the branch: see there)
    while (true) {
        m_run = -INFINITY; l_run = 0.f;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int r = 0; r < 16; ++r) o_acc[dt][r] = 0.f;
        if (RESIDENT) {
            const KernargPtr args = kernarg_block();
            const int index = item_of_round<CAUSAL>(args, bid, ++round);
            has_next = index < args->items;
            q_block = -1;
            if (has_next) {
                nx = locate_item<BN, CAUSAL, SPLIT, true>(args, index);
                q_block = it.nb_end - 2 > it.nb_begin ? it.nb_end - 2 : it.nb_begin;
            }
        }
        if (it.nb_begin < it.nb_end) {
            {
                v4i fr[KS];
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) fr[ks] = *(const v4i*)(smem + (k_rd(ks) + buf * KT));
                sacc = (v16i){0};
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) sacc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fr[ks], qreg[ks], sacc, 0, 0, 0);
            }
            int nb = it.nb_begin;
            if (RESIDENT) {
                const int last = it.nb_end - 1;
                while (true) {
                    if (buf == 0) {
                        if (nb >= last) break;
                        compute(BoolTag<false>{}, 0, nb++);
                        v_here = false;
                    }
                    buf = 1;
                    if (nb >= last) break;
                    compute(BoolTag<false>{}, 1, nb++);
                    v_here = false;
                    buf = 0;
                }
                compute(BoolTag<true>{}, buf, nb);
            } else {
                while (true) {
                    if (nb >= it.nb_end) break;
                    compute(BoolTag<false>{}, 0, nb++);
                    if (nb >= it.nb_end) break;
                    compute(BoolTag<false>{}, 1, nb++);
                }
            }
        }

    // ---- epilogue
    const KernargPtr pe = kernarg_block();
    const int e_heads = pe->heads, e_seqlen = pe->seqlen;
    const int eb = it.b, eh = it.h;
    const int q_row = it.mb * kBlockM + rw * 32 + lq;
    const bool q_valid = q_row < e_seqlen;
    // row sum: this wave's keys plus the partner's (the last block's barriers lie between the last use of the exchange
    // slots and this one)
    float l_tot = half_pair_sum(l_run);          // in units of 1/127 when PROUND == 0
    *(float*)(smem + xm_wr) = l_tot;
    __syncthreads();
    l_tot += *(const float*)(smem + xm_rd);
    if (!RESIDENT && !VBLK) v_scale_bits = load_scale_bits(pe->v_scale, eb * pe->vs_sb + it.hk * pe->vs_sh, pe->scale_dtype);
    asm volatile("" : "+v"(v_scale_bits));       // (arrived here on every way: a load that the compiler takes for pending in the next item makes it wait there)
    const float vs = VBLK ? 1.f : cvt_scale_bits(v_scale_bits, pe->scale_dtype);
    // (a row without a visible key gives zeros and lse = -inf; its accumulators hold NaN from exp2(-inf - -inf), hence
    // the selects)
    const bool any_key = it.nb_begin < it.nb_end && m_run > -INFINITY;
    const float out_scale = !any_key ? 0.f : (PROUND == 0) ? (vs / l_tot) : (vs / (127.f * l_tot));
    const float l_true = (PROUND == 0) ? l_tot * (1.f / 127.f) : l_tot;
    const float lse = any_key ? m_run + __builtin_log2f(l_true) : -INFINITY;
    if (SPLIT) {
        const int64_t row = ((int64_t)(it.split * pe->batch + eb) * e_heads + eh) * e_seqlen + q_row;
        float* op = pe->o_part + row * D + hf * DVW;
        if (q_valid) {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int a4 = 0; a4 < 4; ++a4) {
                    v4f o;
#pragma unroll
                    for (int b4 = 0; b4 < 4; ++b4) o[b4] = any_key ? o_acc[dt][4 * a4 + b4] * out_scale : 0.f;
                    *(v4f*)(op + 32 * dt + 8 * a4 + 4 * lh) = o;
                }
            if (lh == 0 && hf == 0) pe->lse_part[row] = lse;
        }
        return;
    }
    {
    // the next item's first tiles, k_scale and Q have arrived (ahead of the stores)
    if (RESIDENT && has_next) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        asm volatile("" : "+v"(q_scale_bits));
        if (ks_wave) put_ks(ks_next, buf ^ 1);
    }
    // 16-bit rows go out through LDS (whole lines per store instruction): waves 0-3 through the last block's tiles (every wave has
    // passed the barrier of the row-sum exchange, so none of them is read any more)
    // (an opaque copy of the lane index: the staging addresses depend on the lane only and would otherwise be computed
    // ahead of the main loop and held in registers through it)
    int lane_e = lane;
    asm volatile("" : "+v"(lane_e));
    const int lq_e = lane_e & 31, lh_e = lane_e >> 5;
    constexpr int OSB = OutStage<DVW>::BYTES;
    char* const stage = smem + (wave < 2 ? OFF_K + buf * KT + wave * OSB : wave < 4 ? OFF_V + buf * KT + (wave - 2) * OSB : OFF_ST + (wave - 4) * OSB);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int a4 = 0; a4 < 4; ++a4) {
            const int d0 = 32 * dt + 8 * a4 + 4 * lh_e;
            if (OUT_DT == 0) {
                v4h o;
#pragma unroll
                for (int b4 = 0; b4 < 4; ++b4) o[b4] = (_Float16)(any_key ? o_acc[dt][4 * a4 + b4] * out_scale : 0.f);
                out_stage_put<DVW>(stage, lq_e, d0, __builtin_bit_cast(v2i, o));
            } else {
                v4s o;
#pragma unroll
                for (int b4 = 0; b4 < 4; ++b4) o[b4] = f32_to_bf16(any_key ? o_acc[dt][4 * a4 + b4] * out_scale : 0.f);
                out_stage_put<DVW>(stage, lq_e, d0, __builtin_bit_cast(v2i, o));
            }
        }
    const int row0 = it.mb * kBlockM + rw * 32;
    out_stage_flush<DVW>(stage, pe->out + eb * pe->o_sb + eh * pe->o_sh + (int64_t)row0 * pe->o_sn + hf * DVW * 2, pe->o_sn,
                         e_seqlen - row0, lane_e);
    if (q_valid && pe->lse != nullptr && lh == 0 && hf == 0) pe->lse[((int64_t)eb * e_heads + eh) * e_seqlen + q_row] = lse;
    }
    if (!RESIDENT || !has_next) return;
    __syncthreads();
    const uint32_t q_rd0 = OFF_Q + (32 * rw + lq) * D + ((lh ^ k_swz) << 4);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qreg[ks] = *(const v4i*)(smem + (q_rd0 ^ (uint32_t)(32 * ks)));
    qsc = q_scale_log2(p, q_scale_bits);
    it = nx;
    buf ^= 1;
    v_here = true;
    }
#endif  // __HIP_DEVICE_COMPILE__
}

}  // namespace intfa
