// Device-side building blocks shared by the forward kernels (gfx950 / CDNA4 only).
//
// Tile geometry used throughout:
//   * a workgroup is 4 wavefronts (256 threads) and owns BLOCK_M = 128 query rows, 32 per wavefront;
//   * keys are consumed in blocks of 128 or 64 (per kernel and head_dim), each handled as sub-tiles of 32 keys;
//   * the score tile is computed TRANSPOSED, S^T = K Q^T, with v_mfma_i32_32x32x32_i8: a lane then holds one
//     query column (lane % 32) and 16 keys, so row max / row sum are in-lane reductions plus one exchange
//     between lane l and lane l^32, and the accumulator registers run along the key axis - the contraction
//     axis of P V - which lets P be packed to int8 in-lane and fed straight back as an MFMA B operand.
//
// MFMA register layouts relied on (verified on hardware against a CPU matmul):
//   v_mfma_i32_32x32x32_i8   A: lane (m = l%32, h = l/32) holds bytes k = 16h .. 16h+15 of row m
//                            B: lane (n = l%32, h)        holds bytes k = 16h .. 16h+15 of column n
//                            D: lane (n = l%32, h) register r holds row m = 8*(r/4) + 4*h + r%4
//   v_mfma_f32_32x32x16_f16  same with 8 halves per lane, k = 8h .. 8h+7
//   ds_read_b64_tr_b8        inside each group of 16 lanes, result lane i byte j = byte (i%8) of the 8 bytes
//                            addressed by lane (2j + i/8) of the group
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace intfa {

typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef __bf16 v4bf __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef short v4s __attribute__((ext_vector_type(4)));

#define INTFA_LDS(p) ((__attribute__((address_space(3))) void*)(p))
// compile-time switch passed as a lambda argument (selects the LDS buffer or the masked code instance of a pipeline step)
template <bool V> struct BoolTag { static constexpr bool value = V; };
template <int V> struct IntTag { static constexpr int value = V; };
#define INTFA_GLB(p) ((const __attribute__((address_space(1))) void*)(p))

// The wait states between a 32 x 32 matrix product and the first other instruction on its registers, where that instruction stands behind
// branches: the compiler counts along the longer of two ways to it, so that scores and accumulators could be read up to three wait states early by waves
// that skip the products in between (mfma_check.py).
__device__ __forceinline__ void wait_for_product(v16i& x) { asm volatile("s_nop 11" : "+v"(x)); }
__device__ __forceinline__ void wait_for_product(v16f& x) { asm volatile("s_nop 11" : "+v"(x)); }

// Behind the first wait for the tiles: Q was requested with them and has arrived too, and this tells the compiler, which does not know the
// hand-written waits.  Without it its own wait for Q stands ahead of the products inside the loop over the key blocks, behind the requests for the
// next tiles, and waits for those: no copy runs under a block's work then (mfma_check.py looks for such waits).  Without -> with it, us: half-int8
// decode d64 B8 H32 Nq1 Nk4096, one pass, 51.3 -> 37, 320 workgroups of 6000 keys 78 -> 66; 32 rows, fp16, 102 -> 87; bf16 prefill B4 H32 N4096 d128 964 ->
// 935, causal N2048 d256 425 -> 403.
template <int N> __device__ __forceinline__ void q_has_arrived(v4i (&q)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("" : "+v"(q[i]));
}

constexpr int kBlockM = 128;
constexpr int kThreads = 256;
constexpr float kLog2_127 = 6.98868468677f;   // log2(127)
// floor(n / d) for 0 <= n < 2^31 and a divisor d fixed per launch: (n * m) >> s with s = 31 + ceil(log2 d) and
// m = ceil(2^s / d) < 2^32 computed on the host (Granlund & Montgomery, "Division by invariant integers using
// multiplication").  For a wave-uniform n that is three scalar instructions; a run-time integer division expands to some
// forty dependent vector instructions, and the mapping of a workgroup to its work needs a dozen of them.
struct FastDiv { uint32_t m, s; };
__host__ __device__ __forceinline__ int fast_div(int n, FastDiv d) { return (int)(((uint64_t)(uint32_t)n * d.m) >> d.s); }

// Kernel-side parameter block (byte strides, resolved pointers).
struct KParams {
    const char* q; const char* k; const char* v; char* out;
    const char* q_scale; const char* k_scale; const char* v_scale;
    float* lse;
    const int32_t* seqlens_k;              // optional [batch]: number of keys per batch entry (<= seqlen_k)
    int32_t* s_dump;                       // debug: int32 S [B,H,N,N]
    float* o_part; float* lse_part;        // split-KV partials [S,B,H,N,D] fp32 / [S,B,H,N]
    uint64_t* ticket; uint64_t epoch;      // arrival words of the query blocks, the launch's epoch (intfa_splitkv.h); nullptr: no merge here
    int64_t q_sb, q_sh, q_sn;              // bytes
    int64_t k_sb, k_sh, k_sn;
    int64_t v_sb, v_sh, v_sn;
    int64_t o_sb, o_sh, o_sn;
    int64_t qs_sb, qs_sh, qs_sn;           // elements
    int64_t ks_sb, ks_sh, ks_sn;
    int64_t vs_sb, vs_sh;
    int64_t vs_sblk;                       // blocked V scales: elements between the scale rows of consecutive key ranges
    int32_t batch, heads, seqlen, head_dim;  // seqlen = number of query rows
    int32_t seqlen_k;                      // number of keys (= seqlen unless the caller passes separate lengths)
    int32_t scale_dtype, causal, num_splits, blocks_per_split;
    int32_t kv_group;                      // query heads per K/V head (1 = every query head has its own K/V)
    int32_t vs_g;                          // blocked V scales: key blocks of the kernel per scale row (0 = scalar V scale)
    int32_t vs_sub;                        // blocked V scales: 2 when a scale row covers 64 keys, half of the 128-key block
    int32_t causal_rows;                   // decode kernel: query positions per folded query head (0 = the row is the position)
    float qk_scale_log2;                   // sm_scale * log2(e)
    // workgroup -> work mapping of this launch (set by finish_mapping() in intfa_launch.h from the grid size)
    int32_t per_head;                      // workgroups per query head
    int32_t heads_kv;                      // heads / kv_group
    int32_t xcd_whole_wgs;                 // workgroups of the K/V heads that are dealt whole to the 8 XCDs (a multiple of 8)
    int32_t xcd_rem_chunk;                 // the remaining heads: consecutive workgroups per XCD (0: dealt one by one)
    FastDiv d_per_kv, d_heads_kv, d_per_head, d_n_split, d_heads, d_kv_group;
    // causal launches: the K/V heads of an XCD in groups of run_units (the last one run_units_last), query-block-major in each
    int32_t run_units, run_units_last, run_last_slot;      // run_last_slot: first slot of the last group
    int32_t rem_wgs;                                       // workgroups of the K/V heads that are not dealt whole
    int32_t kv_key_bytes;                                  // bytes of one key's K and V rows
    int32_t stream_kv;                                     // decode-shaped kernels: K and V tiles are loaded non-temporally
    FastDiv d_run, d_run_heads, d_run_heads_last, d_rem_heads;
    int32_t items, grid_wgs;               // work items (workgroups, were each to take one), and workgroups of the launch (last: the others keep their places in the lines)
};

// The kernel's own argument block as the epilogues re-read it: the pointer keeps the constant address space, so its
// fields arrive through scalar loads (a generic pointer would make them vector loads that a vmcnt wait has to cover).
typedef const __attribute__((address_space(4))) KParams* KernargPtr;
__device__ __forceinline__ KernargPtr kernarg_block() {
    KernargPtr pe = (KernargPtr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(pe));       // opaque: the fields are loaded where they are used, not held since the prologue
    return pe;
}
// Requests every 64-byte line of the kernel's argument block in one go.  The block is cold in each launch, and a workgroup's prologue
// reads it in three or four places that depend on one another: each would be a trip to memory of its own, ahead of the first tile load.
// The statement passes the workgroup's number through, on which everything else depends.  (Not a volatile one: the compiler would take it
// for a possible write to memory and load what follows through the vector unit.)
__device__ __forceinline__ int block_after_kernargs() {
    int bid = blockIdx.x;
    typedef const __attribute__((address_space(4))) int* Words;
    const Words w = (Words)__builtin_amdgcn_kernarg_segment_ptr();
    static_assert((sizeof(KParams) - 1) / 64 == 7, "the statement names a word of each line");
    asm("" : "+s"(bid) : "s"(w[0]), "s"(w[16]), "s"(w[32]), "s"(w[48]), "s"(w[64]), "s"(w[80]), "s"(w[96]), "s"(w[112]));
    return bid;
}
// A scale as its bits, and their conversion: the request does not wait for the value, so it can stand ahead of work that hides it.
__device__ __forceinline__ uint32_t load_scale_bits(const char* base, int64_t idx, int dtype) {
    if (dtype == 2) return ((const uint32_t*)base)[idx];
    return ((const uint16_t*)base)[idx];
}
__device__ __forceinline__ float cvt_scale_bits(uint32_t raw, int dtype) {
    if (dtype == 0) return (float)__builtin_bit_cast(_Float16, (uint16_t)raw);
    return __builtin_bit_cast(float, dtype == 1 ? raw << 16 : raw);
}
__device__ __forceinline__ float load_scale(const char* base, int64_t idx, int dtype) {
    if (dtype == 0) return (float)((const _Float16*)base)[idx];
    if (dtype == 1) return __builtin_bit_cast(float, ((uint32_t)((const uint16_t*)base)[idx]) << 16);
    return ((const float*)base)[idx];
}

// ---- What every forward kernel does before its main loop: which (batch, head, query block, split) the workgroup
// works on, which key blocks it visits, its Q fragments and scales.  One copy, shared by the four kernels.

// blockIdx.x -> (batch * heads + head, index among the head's `per_head` workgroups).  Workgroups are dealt round-robin to
// the 8 XCDs, each with its own L2: every XCD gets whole K/V heads, so the K/V tiles of a head are re-read from one L2.
// With grouped K/V heads (kv_group query heads share one K/V head) the unit dealt to an XCD is the K/V head: all query
// heads of a group run on the XCD whose L2 holds their K/V.
// When the number of (batch, K/V head) pairs is no multiple of 8, the first 8 * floor(pairs / 8) are dealt whole as above and
// the workgroups of the remaining pairs, taken in head order, are cut into 8 equal runs, one per XCD: a remaining head's
// K/V then reaches two or three L2s instead of all eight.
// Causal launches: query blocks differ in work by a factor of their number, so the order decides how long the last ones run
// alone.  The K/V heads of an XCD are taken in groups of a few rounds of its workgroup slots; inside a group the heaviest
// query blocks of all its heads come first (a head's own blocks one after the other leave the last heads' heavy blocks to the
// end: N 3333, 64 heads on 16 K/V heads, fp16 d128 223 -> 200 us).  The remaining pairs are one such group over all XCDs,
// ahead of the others: their heavy blocks must not come last either.
// (All divisors are fixed per launch: fast_div.)
struct WorkgroupJob { int b, h, hk, rem; };      // batch entry, query head, K/V head, index among the head's workgroups
// (Args: const KParams* or KernargPtr)
template <typename Args> __device__ __forceinline__ WorkgroupJob deal_workgroup(Args p, int bid) {
    const int kv_group = p->kv_group;
    const int per_head = p->per_head;
    const int per_kv = per_head * kv_group;              // workgroups per K/V head
    int kv_lin, hq, rem;
    if (p->causal) {
        int idx, first, unit_step, heads;
        FastDiv d_heads;
        if (bid >= p->rem_wgs) {
            const int slot = (bid - p->rem_wgs) >> 3;
            unit_step = 8;
            if (slot < p->run_last_slot) {
                const int g = fast_div(slot, p->d_run);
                idx = slot - g * p->run_units * per_kv;
                first = g * p->run_units; heads = p->run_units * kv_group; d_heads = p->d_run_heads;
            } else {
                idx = slot - p->run_last_slot;
                first = fast_div(p->run_last_slot, p->d_per_kv); heads = p->run_units_last * kv_group; d_heads = p->d_run_heads_last;
            }
            first = first * 8 + ((bid - p->rem_wgs) & 7);
        } else {
            idx = bid;
            unit_step = 1;
            first = fast_div(p->xcd_whole_wgs, p->d_per_kv);
            heads = (p->batch * p->heads_kv - first) * kv_group; d_heads = p->d_rem_heads;
        }
        rem = fast_div(idx, d_heads);
        const int u = idx - rem * heads, unit = fast_div(u, p->d_kv_group);
        kv_lin = first + unit * unit_step;
        hq = u - unit * kv_group;
    } else {
        int r;
        if (bid < p->xcd_whole_wgs) {
            const int xcd = bid & 7, slot = bid >> 3;
            const int q = fast_div(slot, p->d_per_kv);
            kv_lin = q * 8 + xcd;
            r = slot - q * per_kv;
        } else {
            const int j = bid - p->xcd_whole_wgs;                        // (xcd_whole_wgs is a multiple of 8: j & 7 is the XCD)
            const int idx = p->xcd_rem_chunk ? (j & 7) * p->xcd_rem_chunk + (j >> 3) : j;
            const int q = fast_div(idx, p->d_per_kv);
            kv_lin = fast_div(p->xcd_whole_wgs, p->d_per_kv) + q;
            r = idx - q * per_kv;
        }
        hq = fast_div(r, p->d_per_head);                  // query head inside the group
        rem = r - hq * per_head;
    }
    const int bb = fast_div(kv_lin, p->d_heads_kv), hk = kv_lin - bb * p->heads_kv;
    return {bb, hk * kv_group + hq, hk, rem};
}
__device__ __forceinline__ WorkgroupJob deal_workgroup(const KParams& p, int bid) { return deal_workgroup(&p, bid); }

// Number of keys of batch entry b: one length for all, or per batch (a cache filled to different lengths), clamped to
// [0, seqlen_k] so that rows past the allocation are never addressed.
template <typename Args> __device__ __forceinline__ int keys_of_batch(Args p, int b) {
    int seqlen_k = p->seqlen_k;
    if (p->seqlens_k != nullptr) {
        const int n = p->seqlens_k[b];
        seqlen_k = n < 0 ? 0 : (n < seqlen_k ? n : seqlen_k);
    }
    return seqlen_k;
}
__device__ __forceinline__ int keys_of_batch(const KParams& p, int b) { return keys_of_batch(&p, b); }

// Key blocks [begin, end) of BN keys that a workgroup visits.  `visible_end` is the end of the range before a split
// narrows it (the blocks that hold a key visible to some row of the workgroup).
//   causal: the mask is aligned to the bottom right corner (csrc/mask.h:53,172 of the reference's CUDA tree): the row at
//           position i sees keys 0 .. i + causal_off, causal_off = seqlen_k - (number of positions); pos_end is one past the
//           workgroup's largest position.
//   split_on: with deal_visible the VISIBLE blocks are dealt evenly to the splits (no split of a query block is empty or
//           short); otherwise the blocks of the whole sequence are, blocks_per_split each (csrc/flash_fwd_kernel.h:503-511).
struct KeyBlocks { int total, begin, end, visible_end; };
template <int BN>
__device__ __forceinline__ KeyBlocks key_block_range(int seqlen_k, bool causal, int pos_end, int causal_off, bool split_on, int n_split,
                                                     int split, bool deal_visible, int blocks_per_split) {
    KeyBlocks r;
    r.total = (seqlen_k + BN - 1) / BN;
    r.begin = 0;
    r.end = r.total;
    if (causal) {
        const int e = (pos_end + causal_off + BN - 1) / BN;
        r.end = e < 0 ? 0 : (e < r.total ? e : r.total);
    }
    r.visible_end = r.end;
    if (split_on) {
        const int per = deal_visible ? (r.end + n_split - 1) / n_split : blocks_per_split;
        r.begin = split * per;
        const int e = r.begin + per;
        r.end = e < r.end ? e : r.end;
    }
    return r;
}

// A work item of the general kernels: 128 query rows of one (batch, head), and the key blocks of them (or of one split).
// LATER: an item after a workgroup's first one (launch_resident in intfa_launch.h: all batch entries have the same length there).  Its
// arguments come through an opaque copy of the block's address (Args: KernargPtr), so that they are loaded where they are used and not held in scalar
// registers from the first item on.
struct WorkItem { int b, h, hk, mb, split, seqlen_k, nb_begin, nb_end; };
template <int BN, bool CAUSAL, bool SPLIT, bool LATER, typename Args>
__device__ __forceinline__ WorkItem locate_item(Args args, int index) {
    const WorkgroupJob wg = deal_workgroup(args, index);
    const int n_split = SPLIT ? args->num_splits : 1;
    const int mb_idx = SPLIT ? fast_div(wg.rem, args->d_n_split) : wg.rem;
    WorkItem it;
    it.split = wg.rem - mb_idx * n_split;
    it.mb = CAUSAL ? (args->seqlen + kBlockM - 1) / kBlockM - 1 - mb_idx : mb_idx;       // heaviest query blocks first
    it.b = wg.b; it.h = wg.h; it.hk = wg.hk;
    it.seqlen_k = LATER ? args->seqlen_k : keys_of_batch(args, it.b);
    // causal mask aligned to the bottom right corner: query row i sees keys 0 .. i + (seqlen_k - seqlen)
    const KeyBlocks kb = key_block_range<BN>(it.seqlen_k, CAUSAL, it.mb * kBlockM + kBlockM, it.seqlen_k - args->seqlen, SPLIT, n_split,
                                             it.split, CAUSAL, args->blocks_per_split);
    it.nb_begin = kb.begin; it.nb_end = kb.end;
    return it;
}
// Index of a workgroup's item of the given round (0: its first one), or one past the last item where it has none: every grid-th, and causal
// every second round backwards (the lengths of two rounds then add up to the same in every workgroup).
template <bool CAUSAL> __device__ __forceinline__ int item_of_round(KernargPtr args, int bid, int round) {
    const int grid = args->grid_wgs;
    return round * grid + (CAUSAL && (round & 1) ? grid - 8 - (bid & ~7) + (bid & 7) : bid);      // (bid & 7: the XCD)
}

// int8 Q fragments of query row q_ld (B operand of S^T = K Q^T): 16 bytes per k-step of 32, the half lh of the lane.
template <int KS>
__device__ __forceinline__ void load_q8_fragments(v4i (&qreg)[KS], const KParams& p, int b, int h, int q_ld, int lh) {
    const char* qrow = p.q + b * p.q_sb + h * p.q_sh + (int64_t)q_ld * p.q_sn;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qreg[ks] = *(const v4i*)(qrow + ks * 32 + lh * 16);
}
// q_scale of query row q_ld times sm_scale * log2(e): the factor between S * k_scale and the exponent of exp2.  Never zero: the scores
// of hidden keys are -infinity, and a row of zeros (scale zero, as padding has) must not make NaN of them.  The smallest normal number
// gives a row's visible keys the same exponent as zero would.
__device__ __forceinline__ uint32_t load_q_scale_bits(const KParams& p, int b, int h, int q_ld) {
    return load_scale_bits(p.q_scale, b * p.qs_sb + h * p.qs_sh + (int64_t)q_ld * p.qs_sn, p.scale_dtype);
}
__device__ __forceinline__ float q_scale_log2(const KParams& p, uint32_t bits) {
    const float c = cvt_scale_bits(bits, p.scale_dtype) * p.qk_scale_log2;
    return c == 0.f ? 0x1p-126f : c;
}
__device__ __forceinline__ float load_q_scale_log2(const KParams& p, int b, int h, int q_ld) {
    const float c = load_scale(p.q_scale, b * p.qs_sb + h * p.qs_sh + (int64_t)q_ld * p.qs_sn, p.scale_dtype) * p.qk_scale_log2;
    return c == 0.f ? 0x1p-126f : c;
}

// k_scale of the keys of one (batch, K/V head): fetched as raw bits (one key per thread, ahead of the block that uses
// them) and converted to fp32 when stored to LDS.  Keys past the end read the last key's scale; they are masked later.
struct KScaleSource {
    const char* base;
    int stride, dtype, seqlen_k;
    template <typename Args> __device__ __forceinline__ KScaleSource(Args p, int b, int hk, int seqlen_k_) {
        const int esize = p->scale_dtype == 2 ? 4 : 2;
        base = p->k_scale + (b * p->ks_sb + hk * p->ks_sh) * esize;
        stride = (int)(p->ks_sn * esize);
        dtype = p->scale_dtype;
        seqlen_k = seqlen_k_;
    }
    __device__ __forceinline__ KScaleSource(const KParams& p, int b, int hk, int seqlen_k_) : KScaleSource(&p, b, hk, seqlen_k_) {}
    __device__ __forceinline__ uint32_t load(int key) const {
        key = key < seqlen_k ? key : seqlen_k - 1;
        const char* src = base + (int64_t)key * stride;
        if (dtype == 2) return *(const uint32_t*)src;
        return (uint32_t)*(const uint16_t*)src;
    }
    __device__ __forceinline__ float cvt(uint32_t raw) const {
        if (dtype == 0) return (float)__builtin_bit_cast(_Float16, (uint16_t)raw);
        if (dtype == 1) return __builtin_bit_cast(float, raw << 16);
        return __builtin_bit_cast(float, raw);
    }
};

// The k_scales of a lane's 16 keys of a sub-tile in ONE register: lane i of each row of 16 lanes holds the scale of the lane's i-th key (key
// 8 (i / 4) + 4 lh + i % 4), and a multiplication takes any of them for the whole row with the DPP modifier row_newbcast, at no instruction of its
// own.  (Read as quads of a broadcast address they are a quarter of the wave's LDS reads, of which the CU does one per 3 ns whatever it brings.)
__device__ __forceinline__ uint32_t scale_lane_key(int lane) { return (uint32_t)(8 * ((lane & 15) >> 2) + 4 * (lane >> 5) + (lane & 3)); }
// The i-th of them (a constant once inlined), as an operand of the instruction that uses it.
template <int I> __device__ __forceinline__ float lane_scale_of(float s) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, s), 0x150 + I, 0xf, 0xf, true));
}
__device__ __forceinline__ float lane_scale(float s, int i) {
    switch (i) {
        case 0: return lane_scale_of<0>(s); case 1: return lane_scale_of<1>(s); case 2: return lane_scale_of<2>(s); case 3: return lane_scale_of<3>(s);
        case 4: return lane_scale_of<4>(s); case 5: return lane_scale_of<5>(s); case 6: return lane_scale_of<6>(s); case 7: return lane_scale_of<7>(s);
        case 8: return lane_scale_of<8>(s); case 9: return lane_scale_of<9>(s); case 10: return lane_scale_of<10>(s); case 11: return lane_scale_of<11>(s);
        case 12: return lane_scale_of<12>(s); case 13: return lane_scale_of<13>(s); case 14: return lane_scale_of<14>(s); default: return lane_scale_of<15>(s);
    }
}
// c += f * (the scale of the lane's i-th key).  (Hand-written: the wait states ahead of it, of the product in f and of a vector instruction that writes `scales`,
// are not the compiler's; mfma_check.py looks for them.)
__device__ __forceinline__ void fmac_lane_scale(float& c, float scales, int f, int i) {
    asm("v_fmac_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(c) : "v"(scales), "v"(f), "i"(i));
}
// Int32 scores as fp32 numbers without a conversion: a product chain that starts from the bits of 1.5 * 2^23 instead of zero ends in the bits of
// 1.5 * 2^23 + S (|S| <= 2^22).  With kScoreBias * k_scale subtracted by the multiplication with k_scale, a score takes one instruction instead of two,
// to the same bits where the bias is finite (past_fold): the product is exact inside it, and kScoreBias * k_scale is exact for 16-bit scales (at most 11 + 2 significant bits).
constexpr int kScoreSeed = 0x4B400000;
constexpr float kScoreBias = 12582912.f;
// From 2^104 on (keys of bf16 rows of magnitude 2.6e33 have such scales; infinities) the bias is, or may be, past the largest fp32 number and the
// score would be lost.  A workgroup that meets such a key takes all of its key blocks again with the conversion: the waves that store the
// scales look for them and leave a word in the LDS, which the others read once, behind the last block.
__device__ __forceinline__ bool past_fold(float s) { return __builtin_amdgcn_ballot_w64(__builtin_fabsf(s) >= 0x1p104f) != 0; }

// ---- LDS swizzles.  A tile row is ROW_BYTES bytes; its 16-byte chunks are XOR-permuted with a function of the
// row so that the rows touched together by one LDS access cycle (64 banks x 4 bytes = 256 bytes: 16 lanes of a
// 16-byte read, 32 lanes of an 8-byte read) fall into different bank groups.  Every function depends on the low
// four bits of the row only.
enum { SWZ_K = 0, SWZ_V8 = 1, SWZ_V16 = 2 };
// K / Q style rows: 16 consecutive lanes read the same chunk of 16 consecutive rows.
template <int ROW_BYTES> __device__ __forceinline__ int swz_k(int row) {
    if (ROW_BYTES >= 256) return row & 15;                           // every row starts at bank 0
    if (ROW_BYTES == 128) return (row & 7) ^ ((row >> 3) & 1);       // rows r, r+8 share banks: flip bit 0
    return (row >> 2) & 3;                                           // 64-byte rows: rows r, r+4, r+8, r+12 share banks
}
// int8 V rows read by ds_read_b64_tr_b8: a 16-lane group touches rows {0,1,2,3,8,9,10,11} + 4h of a sub-tile.
template <int ROW_BYTES> __device__ __forceinline__ int swz_v8(int row) {
    // 256-byte rows all start at bank 0, and the two 16-lane groups served together read neighbouring chunks (2 dt and
    // 2 dt + 1) of eight rows each: even flips keep the groups in the even and the odd chunks respectively
    if (ROW_BYTES >= 256) return 2 * ((row & 3) | ((row >> 1) & 4));
    if (ROW_BYTES >= 128) return (row & 3) | ((row >> 1) & 4);
    return ((row >> 1) & 1) | ((row >> 2) & 2);
}
// 16-bit V rows read by ds_read_b64_tr_b16: 32 lanes touch 4 consecutive rows x 64 contiguous bytes.
template <int ROW_BYTES> __device__ __forceinline__ int swz_v16(int row) {
    if (ROW_BYTES >= 256) return (row & 3) << 2;
    return ((row >> 1) & 1) << 2;                                    // 128-byte rows: rows r, r+1 differ by half
}
template <int ROW_BYTES, int SWZ> __device__ __forceinline__ int swz(int row) {
    return SWZ == SWZ_K ? swz_k<ROW_BYTES>(row) : (SWZ == SWZ_V8 ? swz_v8<ROW_BYTES>(row) : swz_v16<ROW_BYTES>(row));
}

// Asynchronous copy of one ROWS-row tile (ROW_BYTES bytes per row) from global memory straight into LDS with
// buffer_load_dwordx4 ... lds: every wave instruction moves 64 x 16 bytes into 1 KiB of consecutive LDS, so the
// swizzle is applied on the GLOBAL side (which chunk a lane fetches).  The four waves split the instructions.
// Addressing is split into a wave-uniform part (SGPRs) and a per-lane 32-bit offset.  The swizzle of a row depends
// on the row's low four bits only; wave w issues instructions w, w+4, w+8, ... whose first rows differ by
// multiples of 4*RPI rows, so a lane needs one offset when 4*RPI >= 16 and 16/(4*RPI) otherwise.
template <int ROW_BYTES, int SWZ, int ROWS> struct TileLoadLane {
    static constexpr int CH = ROW_BYTES / 16;        // 16-byte chunks per row
    static constexpr int RPI = 64 / CH;              // rows per wave instruction
    static constexpr int NINST = ROWS * CH / 64;     // wave instructions per tile
    static constexpr int NV = (4 * RPI >= 16) ? 1 : 16 / (4 * RPI);
    static_assert(CH >= 4 && CH <= 32 && NINST % 4 == 0, "unsupported tile geometry");
    uint32_t off[NV];
};
template <int ROW_BYTES, int SWZ, int ROWS>
__device__ __forceinline__ TileLoadLane<ROW_BYTES, SWZ, ROWS> tile_load_lane(uint32_t row_stride, int wave, int lane) {
    using T = TileLoadLane<ROW_BYTES, SWZ, ROWS>;
    const int rsub = lane / T::CH, cp = lane % T::CH;
    T t;
#pragma unroll
    for (int v = 0; v < T::NV; ++v) {
        const int row = (v * 4 + wave) * T::RPI + rsub;
        const int f = swz<ROW_BYTES, SWZ>(row) & (T::CH - 1);
        t.off[v] = (uint32_t)rsub * row_stride + (uint32_t)((cp ^ f) << 4);
    }
    return t;
}
// The global side is addressed through a buffer resource (base pointer of the (batch, head) slice, SGPRs) plus a
// wave-uniform byte offset (SGPR) plus the lane's 32-bit offset: no 64-bit per-lane pointers.  The copy itself is
// written as inline assembly (M0 = LDS destination of the wave's 1 KiB, then buffer_load_dwordx4 ... lds) so that
// the compiler does not serialise later LDS reads of the OTHER buffer behind it; completion is awaited explicitly
// with s_waitcnt vmcnt(0) before the workgroup barrier that publishes the tile.
__device__ __forceinline__ v4i make_rsrc(const void* base, uint32_t bytes) {
    const uint64_t a = (uint64_t)base;
    v4i r;
    r[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)a);
    r[1] = __builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xffffu));   // stride 0: raw buffer
    r[2] = __builtin_amdgcn_readfirstlane((int)bytes);                              // num_records, bounds-checked
    r[3] = 0x00020000;
    return r;
}
// One wave instruction of a copy: 64 x 16 bytes from the resource at soff + the lane's offset to 1 KiB of LDS.
// The statement overwrites M0 and cannot say so: the compiler keeps M0 reserved on this target, warns about a clobber
// entry for it and ignores it.  Nothing the compiler generates in these kernels reads M0 (no LDS-DMA builtins, GWS,
// relative moves or interpolation), and every copy sets it afresh.  soff and lds must be wave-uniform values
// the compiler can see as such (kernel arguments, readfirstlane results): they end up in scalar operands.
// NT: non-temporal, for tiles that nothing reads again.
template <bool NT> __device__ __forceinline__ void issue_copy_1k(v4i rsrc, uint32_t lane_off, uint32_t soff, uint32_t lds) {
    if (NT) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds"
                 :: "s"(lds), "v"(lane_off), "s"(rsrc), "s"(soff) : "memory");
    else asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :: "s"(lds), "v"(lane_off), "s"(rsrc), "s"(soff) : "memory");
}
// Issues wave instruction number `it` (0 .. NINST/4 - 1) of this wave's share of one tile copy.
template <int ROW_BYTES, int SWZ, int ROWS, bool NT = false>
__device__ __forceinline__ void issue_tile_part(v4i rsrc, uint32_t tile_off, uint32_t row_stride, uint32_t lds_tile,
                                                int wave, const TileLoadLane<ROW_BYTES, SWZ, ROWS>& ln, int it) {
    using T = TileLoadLane<ROW_BYTES, SWZ, ROWS>;
    const int i = it * 4 + wave;                     // wave-uniform instruction index
    const uint32_t m0v = lds_tile + (uint32_t)i * 1024u;
    const uint32_t soff = tile_off + (uint32_t)(i * T::RPI) * row_stride;
    issue_copy_1k<NT>(rsrc, ln.off[it % T::NV], soff, m0v);
}
template <int ROW_BYTES, int SWZ, int ROWS, bool NT = false>
__device__ __forceinline__ void issue_tile_load(v4i rsrc, uint32_t tile_off, uint32_t row_stride, uint32_t lds_tile,
                                                int wave, const TileLoadLane<ROW_BYTES, SWZ, ROWS>& ln) {
    using T = TileLoadLane<ROW_BYTES, SWZ, ROWS>;
#pragma unroll
    for (int it = 0; it < T::NINST / 4; ++it) issue_tile_part<ROW_BYTES, SWZ, ROWS, NT>(rsrc, tile_off, row_stride, lds_tile, wave, ln, it);
}

// ---- 16-bit output rows through LDS.  In the accumulator layout a lane holds four consecutive columns of ONE row per
// register quad, so a direct store writes 8-byte pieces of 32 different rows per instruction and every 64-byte line
// of the output is touched by several partial writes.  Each wave therefore stages its 32 rows x NCOL columns in a
// private LDS region (rows of NCOL * 2 bytes, 16-byte chunks XOR-permuted by the row so that neither the 8-byte
// writes nor the 16-byte reads meet in a bank) and writes them out with 16 bytes per lane: a row's NCOL * 2 bytes are
// contiguous in one store instruction.  The region must be dead tile memory: a workgroup barrier lies between the last
// tile read of any wave and the first out_stage_put.
template <int NCOL> struct OutStage {
    static constexpr int RS = NCOL * 2;                  // bytes per staged row
    static constexpr int CH = RS / 16;                   // 16-byte chunks per row
    static constexpr int RPB = RS >= 256 ? 1 : 256 / RS; // rows per 256 bytes (one pass over the banks)
    static constexpr int BYTES = 32 * RS;                // per wave
    static constexpr int LPR = RS / 16, RPI = 64 / LPR;  // lanes per row / rows per store instruction
    static_assert(NCOL == 64 || NCOL == 128, "staging is laid out for 128- and 256-byte rows");
    static __device__ __forceinline__ int key(int row) { return (row / RPB) & (CH - 1); }
};
// four 16-bit values (columns d0 .. d0 + 3, d0 a multiple of 4) of the wave's row `row`
template <int NCOL>
__device__ __forceinline__ void out_stage_put(char* stage, int row, int d0, v2i bits) {
    using S = OutStage<NCOL>;
    *(v2i*)(stage + row * S::RS + ((((d0 * 2) >> 4) ^ S::key(row)) << 4) + ((d0 * 2) & 15)) = bits;
}
// g_row0: global address of the wave's first row (column offset applied); rows_valid: how many of the 32 rows exist
template <int NCOL>
__device__ __forceinline__ void out_stage_flush(const char* stage, char* g_row0, int64_t row_stride, int rows_valid, int lane) {
    using S = OutStage<NCOL>;
    const int sub = lane / S::LPR, ch = lane % S::LPR;
#pragma unroll
    for (int j = 0; j < 32 / S::RPI; ++j) {
        const int row = j * S::RPI + sub;
        const v4i x = *(const v4i*)(stage + row * S::RS + ((ch ^ S::key(row)) << 4));
        if (row < rows_valid) *(v4i*)(g_row0 + row * row_stride + ch * 16) = x;
    }
}

// fp32 -> bf16 in hardware (v_cvt_pk_bf16_f32 converts two values per instruction, round-to-nearest-even): what the
// attention kernels use for P and for the output.  (The quantisers keep the integer form below: they reproduce another
// library's results bit for bit, NaN patterns included.)
__device__ __forceinline__ short f32_to_bf16(float f) { return __builtin_bit_cast(short, (__bf16)f); }
__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f) {   // round-to-nearest-even
    uint32_t u = __builtin_bit_cast(uint32_t, f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return u >> 16;
}

// Reductions across the two lanes that share a query column (lane l and lane l ^ 32): v_permlane32_swap turns
// one register into (lower halves, upper halves), so one swap plus one max/add serves all 64 lanes.
__device__ __forceinline__ float half_pair_max(float x) {
    const unsigned u = __builtin_bit_cast(unsigned, x);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return fmaxf(__builtin_bit_cast(float, (unsigned)r[0]), __builtin_bit_cast(float, (unsigned)r[1]));
}
__device__ __forceinline__ float half_pair_sum(float x) {
    const unsigned u = __builtin_bit_cast(unsigned, x);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// v for a visible key, -inf for a hidden one (key index k_r past the lane's last visible index `last`), without a
// compare and select: min with a threshold that is +inf or -inf by the sign of last - k_r.  No condition registers,
// so the statement cannot be merged with a wave-uniform test around it into a select per element.
__device__ __forceinline__ float hide_past(float v, int last, int k_r) {
    const uint32_t t = (uint32_t)(last - k_r);
    return __builtin_fminf(v, __builtin_bit_cast(float, (t & 0x80000000u) | 0x7f800000u));
}
// The same for a lane's many keys of a masked block (the general kernels): bit j of hidden_past(last) says that key j of a run of 32 lies past the
// lane's last visible one (`last` may lie before the run or past it), and hide(v, bits, j) is the smaller of v and an infinity with that bit for
// its sign: three instructions where the minimum above takes seven with what the compiler puts around it.  A visible score that is not a number
// becomes +infinity, as there: its row's maximum shows it, also where the row has no other key.  us, causal, minimum -> this: half-int8 d128 B8 H32 N2048
// 286 -> 278, N512 32.2 -> 31.1, full-int8 d128 B4 H32 N4096 432 -> 424, N1024 blocked V scales 39.9 -> 39.6 (with the fold, where it runs).
__device__ __forceinline__ uint32_t hidden_past(int last) {
    const int n = last + 1;
    return (uint32_t)(0xffffffffull << (n < 0 ? 0 : n > 32 ? 32 : n));
}
__device__ __forceinline__ float hide(float v, uint32_t bits, int j) {
    uint32_t m = (uint32_t)__builtin_amdgcn_sbfe((int)bits, (unsigned)j, 1u);
    asm("" : "+v"(m));               // (opaque: else a compare and a select of it)
    const uint32_t most = m << 31 | 0x7f800000u;
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(v), "v"(most));
    return r;
}
// ... and the one that leaves a visible NaN what it is (head_dim 256).
__device__ __forceinline__ float hide_number(float v, uint32_t bits, int j) {
    uint32_t m = (uint32_t)__builtin_amdgcn_sbfe((int)bits, (unsigned)j, 1u);
    asm("" : "+v"(m));
    return __builtin_bit_cast(float, (m & 0xff800000u) | (~m & __builtin_bit_cast(uint32_t, v)));
}

// The reference's requantisation of P (flash_atten_full_int8.py:49-51) for the 16 probabilities a lane holds of one 32-key
// sub-tile: fp16(p) (round to nearest even) * 127 -> fp16, + 0.5 -> fp16, truncating conversion to an integer.  The vector pipe
// bounds the kernels that call this, so the instructions count: 1.75 per value, all but the last packed in pairs.
//   * Product and sum are one packed fma: it skips the rounding of the product, and the truncated result is the same for
//     every fp16 number in [0, 1] (exhaustively: tests/test_p_requant_steps.py).
//   * The truncation is an addition of 1024 with the fp16 rounding mode at "toward zero": the integer lands in the low bits
//     of the mantissa, and one byte permute packs four of them.  (MODE bits 3:2 round fp16 and fp64 results; the statement
//     that sets them restores round-to-nearest, which everything else here runs in.)  NaN gives any byte: its row sum is NaN.
// Before: multiply, add and a converting byte write (SDWA) each, 2.5 per value.  Full-int8, us: d128 B4 H32 N4096 821 -> 793
// (with the fma alone 845 where the old chain took 863), d64 B4 H32 N1024 50.0 -> 47.0, d256 B16 H16 N1024 257 -> 252.
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
// (the same for the 4 NT probabilities of the decode-shaped kernels' lanes: four consecutive keys of NT tiles, four bytes each)
template <int NT> __device__ __forceinline__ void requant_p_reference(const float (&p)[4 * NT], uint32_t (&out)[NT]) {
    unsigned hb[2 * NT];
#pragma unroll
    for (int i = 0; i < 2 * NT; ++i) {
        v2h h = __builtin_convertvector((v2f){p[2 * i], p[2 * i + 1]}, v2h);
        h = __builtin_elementwise_fma(h, (v2h){(_Float16)127.0f, (_Float16)127.0f}, (v2h){(_Float16)0.5f, (_Float16)0.5f});
        hb[i] = __builtin_bit_cast(unsigned, h);
    }
    const unsigned k1024 = 0x64006400u;                    // fp16 1024, twice
    static_assert(NT == 1 || NT == 2, "four or eight probabilities");
    if constexpr (NT == 1)
        asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 2, 2), 3\n\tv_pk_add_f16 %0, %0, %2\n\tv_pk_add_f16 %1, %1, %2\n\t"
                     "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 2, 2), 0" : "+v"(hb[0]), "+v"(hb[1]) : "s"(k1024));
    else
        asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 2, 2), 3\n\tv_pk_add_f16 %0, %0, %4\n\tv_pk_add_f16 %1, %1, %4\n\t"
                     "v_pk_add_f16 %2, %2, %4\n\tv_pk_add_f16 %3, %3, %4\n\ts_setreg_imm32_b32 hwreg(HW_REG_MODE, 2, 2), 0"
                     : "+v"(hb[0]), "+v"(hb[1]), "+v"(hb[2]), "+v"(hb[3]) : "s"(k1024));
#pragma unroll
    for (int t = 0; t < NT; ++t) out[t] = __builtin_amdgcn_perm(hb[2 * t + 1], hb[2 * t], 0x06040200u);
}
__device__ __forceinline__ v4i requant_p_reference16(const float (&p)[16]) {
    unsigned hb[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        v2h h = __builtin_convertvector((v2f){p[2 * i], p[2 * i + 1]}, v2h);
        h = __builtin_elementwise_fma(h, (v2h){(_Float16)127.0f, (_Float16)127.0f}, (v2h){(_Float16)0.5f, (_Float16)0.5f});
        hb[i] = __builtin_bit_cast(unsigned, h);
    }
    const unsigned k1024 = 0x64006400u;                    // fp16 1024, twice
    asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 2, 2), 3\n\t"
                 "v_pk_add_f16 %0, %0, %8\n\tv_pk_add_f16 %1, %1, %8\n\tv_pk_add_f16 %2, %2, %8\n\tv_pk_add_f16 %3, %3, %8\n\t"
                 "v_pk_add_f16 %4, %4, %8\n\tv_pk_add_f16 %5, %5, %8\n\tv_pk_add_f16 %6, %6, %8\n\tv_pk_add_f16 %7, %7, %8\n\t"
                 "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 2, 2), 0"
                 : "+v"(hb[0]), "+v"(hb[1]), "+v"(hb[2]), "+v"(hb[3]), "+v"(hb[4]), "+v"(hb[5]), "+v"(hb[6]), "+v"(hb[7]) : "s"(k1024));
    v4i r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = (int)__builtin_amdgcn_perm(hb[2 * i + 1], hb[2 * i], 0x06040200u);
    return r;
}

}  // namespace intfa
