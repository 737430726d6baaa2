// Host-side launch functions, one per (variant, head_dim), each defined in its own translation unit so that the
// kernel instances compile in parallel.
#pragma once
#include "intfa_device.h"

namespace intfa {

// The MI355X as one device: 8 XCDs of 32 compute units.  The mapping of workgroups to XCDs and the lines between kernels are laid out for
// it; on a partition of the card with fewer of either, the lines lie too high and the order is less even, with the same results.
// (intfa_fwd_suggest_splits takes the device's number from its caller, because a split count may change the results.)
constexpr int kXcds = 8, kCusPerXcd = 32, kComputeUnits = kXcds * kCusPerXcd;

constexpr int kDecodeMaxRows = 64;    // most query rows per head of a decode-shaped call
constexpr int kDecodeRows = 32;       // query rows per workgroup of the decode-shaped kernel (intfa_fwd_decode.h, intfa_fwd_decode_f16pv.h)

// Launch switches resolved to template arguments inside the instance files.
struct LaunchSel {
    bool causal;
    int io_dt;       // 0 fp16, 1 bf16 (type of out; also of V / fp Q,K where those are 16-bit)
    int p_round;     // full-int8 only
    bool split;      // write split-KV partials instead of the output
    bool dump_s;     // full-int8 only: export int32 S and stop
    bool wide;       // decode-shaped kernels: few query rows per head (intfa_fwd_decode_wide.h)
    int row_tiles;   // ... tiles of 16 query rows per workgroup
    bool crowded;    // ... full-int8: more workgroups than the form with the longer pipeline has room for
};

inline FastDiv make_fast_div(int d) {
    int l = 0;
    while ((1ll << l) < (long long)d) ++l;                   // ceil(log2 d), d >= 1
    const unsigned s = 31u + (unsigned)l;
    const unsigned long long m = ((1ull << s) + (unsigned long long)d - 1) / (unsigned long long)d;   // < 2^32
    return {(uint32_t)m, (uint32_t)s};
}
// Fills the workgroup -> work mapping of a launch of `grid` workgroups (grid = batch * heads * workgroups per head).
inline KParams finish_mapping(const KParams& kp, int grid) {
    KParams k = kp;
    const int n_split = kp.num_splits > 1 ? kp.num_splits : 1;
    k.items = k.grid_wgs = grid;
    k.per_head = grid / (kp.batch * kp.heads);
    k.heads_kv = kp.heads / kp.kv_group;
    const int per_kv = k.per_head * kp.kv_group, units = kp.batch * k.heads_kv;
    k.xcd_whole_wgs = (units / kXcds) * kXcds * per_kv;
    k.rem_wgs = grid - k.xcd_whole_wgs;
    k.xcd_rem_chunk = ((units % kXcds) * per_kv) % kXcds == 0 ? (units % kXcds) * per_kv / kXcds : 0;
    // Causal: groups of K/V heads with two rounds of an XCD's workgroup slots (32 compute units; two workgroups each, four at
    // head_dim 64; four rounds at head_dim 256, one each) whose K and V come to 9 MB at most, since all of a group's heads are read at
    // once.  Larger groups lose to the 4 MB L2 (half-int8 B8 H32 N2048 d128: 298 us up to 12 MB, 313 us at 48), smaller ones end
    // unevenly (full-int8 B4 H32 N4096 d64: 390 us with two heads, 349 with eight).
    const int xcd_units = units / kXcds, slots = 2 * kCusPerXcd * (kp.head_dim == 64 ? 4 : 2);
    const int by_slots = slots / per_kv, by_bytes = (int)(9000000 / ((int64_t)kp.seqlen_k * kp.kv_key_bytes));
    int run_units = by_slots < by_bytes ? by_slots : by_bytes;
    run_units = run_units < xcd_units ? run_units : xcd_units;
    k.run_units = run_units > 1 ? run_units : 1;
    const int runs = xcd_units / k.run_units > 0 ? xcd_units / k.run_units : 1;
    k.run_units_last = xcd_units - (runs - 1) * k.run_units;
    if (k.run_units_last < 1) k.run_units_last = 1;
    k.run_last_slot = (runs - 1) * k.run_units * per_kv;
    k.d_run = make_fast_div(k.run_units * per_kv);
    k.d_run_heads = make_fast_div(k.run_units * kp.kv_group);
    k.d_run_heads_last = make_fast_div(k.run_units_last * kp.kv_group);
    k.d_rem_heads = make_fast_div(units % kXcds > 0 ? (units % kXcds) * kp.kv_group : 1);
    k.d_per_kv = make_fast_div(k.per_head * kp.kv_group);
    k.d_heads_kv = make_fast_div(k.heads_kv);
    k.d_per_head = make_fast_div(k.per_head);
    k.d_n_split = make_fast_div(n_split);
    k.d_heads = make_fast_div(kp.heads);
    k.d_kv_group = make_fast_div(kp.kv_group);
    return k;
}

// One workgroup per (batch, head, 128-row query block, split).
template <typename K> inline int launch_kernel(K kernel, const KParams& kp, hipStream_t stream, int threads = kThreads) {
    const int grid = kp.batch * kp.heads * ((kp.seqlen + kBlockM - 1) / kBlockM) * kp.num_splits;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads), 0, stream, finish_mapping(kp, grid));
    return (int)hipGetLastError();
}
// Causal items differ in length, and each of `slots` resident workgroups has a fixed list of them (item_of_round): true if there are two rounds of them
// and no list is longer than the mean by more than a quarter of an item, and a shortest item where they do not come out even: about what the
// hardware's dealing of single ones leaves.  (Full-int8
// head_dim 256, us, dealt by the hardware -> lists: 12 heads of 6000 keys, whose longest list is a third over the mean, 199 -> 248; 8 heads of 6000,
// 1.5 rounds, 150.7 -> 153.0; 192 heads of 500 47.0 -> 43.4, 24 heads of 3000 119.3 -> 115.7.)  Past 32 rounds it is taken for true.
inline bool lists_agree(const KParams& kp, int slots) {
    const int n_mblk = (kp.seqlen + kBlockM - 1) / kBlockM;
    const KParams k = finish_mapping(kp, kp.batch * kp.heads * n_mblk);
    const int lists = slots / kXcds, per_xcd = k.xcd_whole_wgs / kXcds;
    if (k.rem_wgs != 0 || lists > 64 || per_xcd < 2 * lists) return false;
    if (per_xcd >= 32 * lists) return true;
    const int xcd_units = per_xcd / (n_mblk * kp.kv_group);
    int64_t load[64] = {}, total = 0;
    int list = 0, step = 1;                                       // (to and fro: every second round backwards)
    for (int unit = 0; unit < xcd_units;) {
        const int units = unit * n_mblk * kp.kv_group < k.run_last_slot ? k.run_units : k.run_units_last;
        for (int m = n_mblk; m > 0; --m)
            for (int head = 0; head < units * kp.kv_group; ++head) {
                const int64_t keys = (int64_t)m * kBlockM + (kp.seqlen_k - kp.seqlen);
                load[list] += keys;
                total += keys;
                list += step;
                if (list < 0 || list == lists) { step = -step; list += step; }
            }
        unit += units;
    }
    int64_t most = 0;
    for (int i = 0; i < lists; ++i) most = load[i] > most ? load[i] : most;
    const int64_t shortest = kBlockM + (kp.seqlen_k - kp.seqlen);
    return most - total / lists <= total / per_xcd / 4 + (per_xcd % lists != 0 ? shortest : 0);
}
// The same work items for `slots` workgroups (a multiple of kXcds), which take every slots-th each, where there are more items than that.
// Not for batches of different lengths (the items of a workgroup would differ in work; the hardware deals single ones as compute units
// become free), for items that may have no key, or for query rows further apart than a copy's offsets reach.
// (The lists are fixed: a compute unit is held until its list ends, and beside another stream's kernels a workgroup that starts late runs all of its items late.
// Full-int8 head_dim 256 B16 H16 N1024, twenty launches beside as much other work on a second stream, ms, until both have ended, dealt singly -> lists:
// 256 MiB copies 10.0 -> 6.9, fp16 decodes 10.9 -> 9.6, d128 prefills 10.3 -> 10.1, the same again 10.5 -> 10.1; small prefills that leave most units idle,
// which now wait for a launch's end instead of an item's, 8.2 -> 9.8, the twenty launches themselves 6.6 -> 5.6.)
inline bool takes_resident(const KParams& kp, int slots) {
    const int64_t items = (int64_t)kp.batch * kp.heads * ((kp.seqlen + kBlockM - 1) / kBlockM);
    return items > slots && kp.num_splits <= 1 && kp.seqlens_k == nullptr && kp.seqlen_k > 0 && !(kp.causal && kp.seqlen_k < kp.seqlen) &&
           kp.q_sn < (1ll << 31) / kBlockM && (!kp.causal || lists_agree(kp, slots));
}
template <typename K> inline int launch_resident(K kernel, const KParams& kp, hipStream_t stream, int threads, int slots) {
    KParams k = finish_mapping(kp, kp.batch * kp.heads * ((kp.seqlen + kBlockM - 1) / kBlockM));
    k.grid_wgs = slots;
    hipLaunchKernelGGL(kernel, dim3(slots), dim3(threads), 0, stream, k);
    return (int)hipGetLastError();
}

#define INTFA_DECL_LAUNCH(name) int name(const KParams& kp, const LaunchSel& sel, hipStream_t stream)
INTFA_DECL_LAUNCH(launch_full_int8_d64);
INTFA_DECL_LAUNCH(launch_full_int8_d128);
INTFA_DECL_LAUNCH(launch_full_int8_d256);
INTFA_DECL_LAUNCH(launch_full_int8_vblk_d64);     // per-block, per-channel V scales
INTFA_DECL_LAUNCH(launch_full_int8_vblk_d128);
INTFA_DECL_LAUNCH(launch_full_int8_vblk_d256);
INTFA_DECL_LAUNCH(launch_full_int8_vblk64_d128);  // V scale rows of 64 keys (two per 128-key block)
INTFA_DECL_LAUNCH(launch_decode_full_int8_d64);    // few query rows per head: the waves of a workgroup share the keys
INTFA_DECL_LAUNCH(launch_decode_full_int8_d128);
INTFA_DECL_LAUNCH(launch_decode_full_int8_d256);
INTFA_DECL_LAUNCH(launch_decode_half_int8_d64);     // (intfa_fwd_decode_f16pv.h)
INTFA_DECL_LAUNCH(launch_decode_half_int8_d128);
INTFA_DECL_LAUNCH(launch_decode_half_int8_d256);
INTFA_DECL_LAUNCH(launch_decode_fp16_d64);
INTFA_DECL_LAUNCH(launch_decode_fp16_d128);
INTFA_DECL_LAUNCH(launch_decode_fp16_d256);
INTFA_DECL_LAUNCH(launch_half_int8_d64);
INTFA_DECL_LAUNCH(launch_half_int8_d128);
INTFA_DECL_LAUNCH(launch_half_int8_d256);
INTFA_DECL_LAUNCH(launch_fp16_d64);
INTFA_DECL_LAUNCH(launch_fp16_d128);
INTFA_DECL_LAUNCH(launch_fp16_d256);

}  // namespace intfa
