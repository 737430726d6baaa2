// Merge of split-KV partial results (algorithm of csrc/flash_fwd_kernel.h:1212-1235 and :1264-1283 in the
// reference, evaluated in base 2 because the forward kernels keep log2-domain statistics): inside the forward kernel by
// the workgroup that finishes a query block last, or, for callers whose workspace has no room for the arrival tickets, by a
// kernel of its own.
#pragma once
#include "intfa_device.h"

namespace intfa {

// ---- Merge inside the forward kernel.
// A merge kernel costs a decoding step 3.4 - 8 us of GPU time and 3.7 us of host time for its launch, half as much as the
// pass itself.  Instead every workgroup publishes its partial and takes a ticket of its query block; the one that draws the
// last ticket merges the block while the other workgroups of the launch still run.
//   * Partials are written and read at agent scope (sc1: past the L2 of the XCD, which is not coherent with the seven
//     others): each access is what an atomic one at that scope compiles to, so the caches need no write-back and no invalidation.  The
//     ticket is an atomic at the same scope, drawn after the writes have been acknowledged; the merge's loads are held behind it by
//     a fence that orders the compiler and the wave's own issue only (at agent scope it would invalidate the L1 in front of the merge:
//     decoding steps and chunks 1 - 4 % slower, half-int8 drafts d64 14.2 -> 14.8 us, causal chunk 109 -> 112).
//   * A ticket word is the launch's epoch (upper 56 bits, never the same twice in a process) and the arrivals so far.  The
//     workspace is not cleared: every workgroup of the block looks at the word when it starts and exchanges anything that
//     is not of this epoch for (epoch, 0) - under the first tiles' way from HBM, so that the arrival itself is one atomic add
//     (a compare-and-swap loop there, with all splits of a block arriving together, cost 5 us with eight of them).  The last
//     arrival stores zero, so the replays of a captured graph, whose epoch is a constant, find no word of an earlier one.
//   * Each word has 256 bytes to itself: atomics on one line follow one another at some 80 ns, and the words of eight heads side by side
//     made 32 splits of each wait 2.5 - 3.2 us for their tickets (0.5 - 0.6 alone).
constexpr int kTicketStride = 32;              // words
constexpr int kSplitAux = 16;                  // sc1 in the cache-policy operand of the buffer intrinsics
typedef __amdgpu_buffer_rsrc_t BufferRsrc;
typedef unsigned v4u __attribute__((ext_vector_type(4)));

// The partials from row `first` (wave-uniform) of the [split][batch][head][row] axis onward.  A writer starts at its own
// workgroup's first row; the merge addresses all of them from row 0 (the host gives tickets only when they span less than 4 GiB).
struct SplitPartials {
    BufferRsrc o, l;
    uint32_t rows;                             // batch * heads * seqlen: rows of one split
    // (P: KParams pointer, or the kernel-argument pointer of the epilogues)
    template <typename P> __device__ __forceinline__ explicit SplitPartials(P p, int D, int64_t first) {
        rows = (uint32_t)(p->batch * p->heads) * (uint32_t)p->seqlen;
        const int64_t left = (int64_t)rows * p->num_splits - first, ob = left * D * 4, lb = left * 4;
        o = __builtin_amdgcn_make_buffer_rsrc(p->o_part + first * D, 0, (int)(uint32_t)(ob < 0xffffffffll ? ob : 0xffffffffll), 0x00020000);
        l = __builtin_amdgcn_make_buffer_rsrc(p->lse_part + first, 0, (int)(uint32_t)(lb < 0xffffffffll ? lb : 0xffffffffll), 0x00020000);
    }
    __device__ __forceinline__ void put(uint32_t row, int D, int col, v4f x) const {
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, x), o, (row * (uint32_t)D + (uint32_t)col) * 4u, 0, kSplitAux);
    }
    __device__ __forceinline__ void put_lse(uint32_t row, float x) const {
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, x), l, row * 4u, 0, kSplitAux);
    }
    __device__ __forceinline__ v4f get(uint32_t row, int D, int col) const {
        return __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(o, (row * (uint32_t)D + (uint32_t)col) * 4u, 0, kSplitAux));
    }
    __device__ __forceinline__ float get_lse(uint32_t row) const {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(l, row * 4u, 0, kSplitAux));
    }
};

template <int OUT_DT> __device__ __forceinline__ void store_out4(char* dst, v4f acc) {
    if (OUT_DT == 0) {
        v4h o;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = (_Float16)acc[i];
        *(v4h*)dst = o;
    } else {
        v4s o;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = f32_to_bf16(acc[i]);
        *(v4s*)dst = o;
    }
}

// Thread 0, at the start: the ticket word of query block `group` becomes this epoch's.
__device__ __forceinline__ void splitkv_open_tickets(const KParams& p, int group) {
    uint64_t* t = p.ticket + group * kTicketStride;
    uint64_t seen = __hip_atomic_load(t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((seen ^ p.epoch) >= 256u)
        __hip_atomic_compare_exchange_strong(t, &seen, p.epoch, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The same in two halves, for a kernel that has something to do under the look's way to memory and back: thread 0 looks at the word early ...
__device__ __forceinline__ uint64_t splitkv_look_at_tickets(const KParams& p, int group) {
    uint64_t seen = 0;
    if (p.ticket != nullptr && threadIdx.x == 0) seen = __hip_atomic_load(p.ticket + group * kTicketStride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return seen;
}
// ... and exchanges it before its own arrival (one that was exchanged by another workgroup since is left alone).
__device__ __forceinline__ void splitkv_open_tickets(KernargPtr p, int group, uint64_t seen) {
    uint64_t* const t = p->ticket;
    const uint64_t epoch = p->epoch;
    if (t != nullptr && threadIdx.x == 0 && (seen ^ epoch) >= 256u)
        __hip_atomic_compare_exchange_strong(t + group * kTicketStride, &seen, epoch, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Takes this workgroup's ticket of query block `group`; true for the last of the block's num_splits workgroups.
// Called by every thread of the workgroup after its stores; `smem` is free.  Its first kArrivalBytes carry the answer, and no barrier follows
// the reading of it: a wave may read it while another is in the merge already, which therefore leaves these bytes alone.
constexpr int kArrivalBytes = 16;
__device__ __forceinline__ bool splitkv_last_arrival(KernargPtr p, char* smem, int group) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // this wave's partials have reached the point of coherence
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t* t = p->ticket + group * kTicketStride;
        const uint64_t before = __hip_atomic_fetch_add(t, (uint64_t)1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool last = before == (p->epoch | (uint64_t)(p->num_splits - 1));
        if (last) __hip_atomic_store(t, (uint64_t)0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *(int*)smem = last;
    }
    __syncthreads();
    const bool last = __builtin_amdgcn_readfirstlane(*(const int*)smem) != 0;
    if (last) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    return last;
}

// ---- The same for the general full-int8 kernel, whose waves own 32 query rows each: a ticket per wave and no barrier.  The wave
// that arrives last reads the partials in the layout of its accumulators, so the row statistics are one value per lane.
// Instead of a second launch of splitkv_combine_kernel, whose arithmetic and order of splits it keeps (the same bits, whichever
// wave is last), us: causal chunk B2 H32/8 Nq512 Nk7680 d128 (2 splits) 113 -> 105.5, B4 H12/3 Nq300 Nk3000 (4) 47 -> 43.4, d64 H16/4
// Nq600 Nk4000 (7) 35.4 -> 31.1.  Not at head_dim 256, whose rows are spread over two waves.
__device__ __forceinline__ bool splitkv_last_arrival_wave(KernargPtr p, int group) {
    unsigned drew_last = 0;                                // (after the wave's partials have been acknowledged)
    if ((threadIdx.x & 63) == 0) {
        uint64_t* t = p->ticket + group * kTicketStride;
        const uint64_t before = __hip_atomic_fetch_add(t, (uint64_t)1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        drew_last = before == (p->epoch | (uint64_t)(p->num_splits - 1));
        if (drew_last) __hip_atomic_store(t, (uint64_t)0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const bool last = __builtin_amdgcn_readfirstlane(drew_last) != 0;
    if (last) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    return last;
}
// Offset (floats) of a lane's four columns 8 c + 4 lh .. of accumulator quad c inside its wave's block of `nr` rows.  With tickets a
// quad of the wave is one contiguous piece (rows side by side, 16 bytes each): a piece per row wrote and read 32 bytes of every
// line (d64 B3 H16 Nq256 Nk2500 40 us).  Without, rows as splitkv_combine_kernel reads them.
struct WavePartialLayout {
    uint32_t lane, quad;
    __device__ __forceinline__ WavePartialLayout(bool tickets, int D, int nr, int row, int lh) {
        lane = tickets ? (uint32_t)(lh * nr + row) * 4u : (uint32_t)(row * D + 4 * lh);
        quad = tickets ? 8u * (uint32_t)nr : 8u;
    }
};
// acc[dt][4 a4 + b4], quad 4 dt + a4: the merged row.  `block`: first row of the wave's block of nr rows on the row axis of one split; `w`: 1 KiB
// of LDS of this wave.  Returns the merged lse.  The partial of the next split is on its way while one is added, half a row at
// a time.  (The wave's own partial is read back like the others: kept in registers beside sum and loads it spills 100 of them.)
template <int D, typename P>
__device__ __forceinline__ float splitkv_merge_wave(P p, float* w, float (&acc)[D / 32][16], uint32_t block, int nr, int lq, int lh) {
    constexpr int DT = D / 32, H = DT / 2;
    const SplitPartials part(p, D, 0);
    const int ns = p->num_splits, rl = lq < nr ? lq : nr - 1;
    const WavePartialLayout at(true, D, nr, rl, lh);
    v4f x[DT][4];
    auto request = [&](int s, int half) __attribute__((always_inline)) {
        const uint32_t base = ((uint32_t)s * part.rows + block) * (uint32_t)D + at.lane;
#pragma unroll
        for (int dt = half * H; dt < half * H + H; ++dt)
#pragma unroll
            for (int a4 = 0; a4 < 4; ++a4) x[dt][a4] = part.get(0, D, (int)(base + (uint32_t)(4 * dt + a4) * at.quad));
    };
    request(0, 0);
    request(0, 1);
    float l[8];
    auto load8 = [&](int s0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 8; ++u) l[u] = part.get_lse((uint32_t)(s0 + u < ns ? s0 + u : ns - 1) * part.rows + block + (uint32_t)rl);
#pragma unroll
        for (int u = 0; u < 8; ++u) l[u] = s0 + u >= ns ? -INFINITY : l[u];
    };
    float mx = -INFINITY, sum = 0.f;
    for (int s0 = 0; s0 < ns; s0 += 8) {
        load8(s0);
#pragma unroll
        for (int u = 0; u < 8; ++u) mx = fmaxf(mx, l[u]);
    }
    const bool empty = mx == -INFINITY;
    if (empty) mx = 0.f;
    for (int s0 = 0; s0 < ns; s0 += 8) {
        if (ns > 8) load8(s0);
#pragma unroll
        for (int u = 0; u < 8; ++u) sum += fast_exp2(l[u] - mx);
    }
    const float lse = empty ? -INFINITY : __builtin_log2f(sum) + mx;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[dt][r] = 0.f;
    for (int s0 = 0; s0 < ns; s0 += 8) {
        if (ns > 8) load8(s0);
#pragma unroll
        for (int u = 0; u < 8; ++u) w[u * 32 + lq] = empty ? 0.f : fast_exp2(l[u] - lse);       // (both halves of the wave write the same)
        const int s_end = s0 + 8 < ns ? s0 + 8 : ns;
        for (int s = s0; s < s_end; ++s) {
            const float ws = w[(s - s0) * 32 + lq];
            const int s_next = s + 1;
#pragma unroll
            for (int half = 0; half < 2; ++half) {
#pragma unroll
                for (int dt = half * H; dt < half * H + H; ++dt)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[dt][r] = fmaf(ws, x[dt][r >> 2][r & 3], acc[dt][r]);
                if (s_next < ns) request(s_next, half);
            }
        }
    }
    return lse;
}

// The four lanes l, l ^ 16, l ^ 32, l ^ 48; the sixteen lanes of a row of 16; all lanes of the wave.
template <typename F> __device__ __forceinline__ float reduce_row_lanes(float x, F op) {
    const unsigned u = __builtin_bit_cast(unsigned, x);
    const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const float y = op(__builtin_bit_cast(float, (unsigned)a[0]), __builtin_bit_cast(float, (unsigned)a[1]));
    const unsigned w = __builtin_bit_cast(unsigned, y);
    const auto c = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    return op(__builtin_bit_cast(float, (unsigned)c[0]), __builtin_bit_cast(float, (unsigned)c[1]));
}
// Of two values at once: lanes of even rows of 16 return the maximum of a over their four lanes, those of odd rows that of b.
__device__ __forceinline__ float max_of_row_lanes(float a, float b) {
    const auto s = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
    const unsigned w = __builtin_bit_cast(unsigned, fmaxf(__builtin_bit_cast(float, (unsigned)s[0]), __builtin_bit_cast(float, (unsigned)s[1])));
    const auto c = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    return fmaxf(__builtin_bit_cast(float, (unsigned)c[0]), __builtin_bit_cast(float, (unsigned)c[1]));
}
template <typename F> __device__ __forceinline__ float reduce_wave(float x, F op) {      // (quad_perm 1,0,3,2 / 2,3,0,1, the mirrored half row, the mirrored row)
    x = op(x, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0xB1, 0xf, 0xf, true)));
    x = op(x, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x4E, 0xf, 0xf, true)));
    x = op(x, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x141, 0xf, 0xf, true)));
    x = op(x, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x140, 0xf, 0xf, true)));
    return reduce_row_lanes(x, op);
}

constexpr int kMaxSplits = 64;                           // the lanes of a wave
constexpr int kMergeWaves = 8;
constexpr int kMergeLds = kArrivalBytes + kMergeWaves * 64 * 16;      // of the workgroup's LDS, from its first byte

// More rows than waves: a wave takes four rows at a time, so that the chains of their weights run side by side, and D / 4 lanes a row of the
// sums; partials of the next four splits are on their way while four are added.  Row after row, as below, the chains were 0.25 us
// each: 32 rows, full-int8 d64 B9 H8 Nq32 Nk9000 27.0 -> 24, fp16 d64 B5 H32/8 Nq6 Nk7000 18.9 -> 18.3 us.
template <int D, int OUT_DT, int WAVES, typename P>
__device__ __forceinline__ void splitkv_merge_many(P p, const SplitPartials& part, char* smem, uint32_t base, char* out0, int nrows, int ns, int wave, int lane) {
    constexpr int LPR = D / 4, SUBS = 64 / LPR, U = 4, C = 4;      // C rows side by side
    const int sub = lane / LPR, col = (lane % LPR) * 4, groups = (ns + U - 1) / U;
    float* const ws = (float*)(smem + kArrivalBytes) + wave * (C * 64);      // weights of the wave's rows, of no other wave's concern
    static_assert(kArrivalBytes + WAVES * C * 64 * 4 <= kMergeLds, "");
    for (int first = wave; first < nrows; first += C * WAVES) {      // rows first, first + WAVES, ...
        auto row_of = [&](int i) __attribute__((always_inline)) { const int r = first + WAVES * i; return r < nrows ? r : first; };
        float lse[C], mx[C], total[C];
#pragma unroll
        for (int i = 0; i < C; ++i) lse[i] = part.get_lse((uint32_t)(lane < ns ? lane : ns - 1) * part.rows + base + (uint32_t)row_of(i));
        v4f x[U], y[U];
        auto request = [&](v4f (&v)[U], int pass, int g) __attribute__((always_inline)) {
            const uint32_t row = base + (uint32_t)row_of(pass * SUBS + sub);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int s = g * U + u;
                v[u] = part.get((uint32_t)(s < ns ? s : ns - 1) * part.rows + row, D, col);
            }
        };
        request(x, 0, 0);
        bool empty[C];                                     // a row no split saw a key for: zeros with lse = -inf, as in splitkv_combine_kernel
#pragma unroll
        for (int i = 0; i < C; ++i) {
            lse[i] = lane < ns ? lse[i] : -INFINITY;
            mx[i] = reduce_wave(lse[i], [](float a, float c) { return fmaxf(a, c); });
            empty[i] = mx[i] == -INFINITY;
            if (empty[i]) mx[i] = 0.f;
        }
#pragma unroll
        for (int i = 0; i < C; ++i) {
            total[i] = reduce_wave(fast_exp2(lse[i] - mx[i]), [](float a, float c) { return a + c; });
            total[i] = empty[i] ? -INFINITY : __builtin_log2f(total[i]) + mx[i];
            ws[64 * i + lane] = empty[i] ? 0.f : fast_exp2(lse[i] - total[i]);      // lane s: the weight of split s (0 past the last one)
            if (p->lse != nullptr && lane == 0 && first + WAVES * i < nrows) p->lse[base + first + WAVES * i] = total[i];
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        const v4f zero = {0.f, 0.f, 0.f, 0.f};
        v4f acc[U] = {zero, zero, zero, zero};             // (four sums, the order of splitkv_merge_rows at head_dim 64)
        int pass = 0, g = 0;
        auto add = [&](const v4f (&v)[U]) __attribute__((always_inline)) {
            const v4f w = *(const v4f*)(ws + 64 * (pass * SUBS + sub) + g * U);
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[u][i] = fmaf(w[u], v[u][i], acc[u][i]);
            if (++g < groups) return;
            const int r = first + WAVES * (pass * SUBS + sub);
            if (r < nrows) store_out4<OUT_DT>(out0 + (int64_t)r * p->o_sn + col * 2, (acc[0] + acc[1]) + (acc[2] + acc[3]));
#pragma unroll
            for (int u = 0; u < U; ++u) acc[u] = zero;
            g = 0;
            ++pass;
        };
        constexpr int PASSES = C / SUBS;
        auto request_next = [&](v4f (&v)[U]) __attribute__((always_inline)) {
            const bool wrap = g + 1 == groups;
            if (!wrap || pass + 1 < PASSES) request(v, wrap ? pass + 1 : pass, wrap ? 0 : g + 1);
        };
        while (true) {
            request_next(y);
            add(x);
            if (pass == PASSES) break;
            request_next(x);
            add(y);
            if (pass == PASSES) break;
        }
    }
}

// Merges the `nrows` (at most 32) rows from row0 of (b, h) out of the partials; WAVES waves, kMergeLds bytes of `smem` (those behind the
// first kArrivalBytes).
// This runs once, at the end of a query block, and its time is a chain of latencies: a wave takes a row, its lanes the row's log-sum-exps
// (lane s that of split s), which make the weights without a word of LDS, and the partials of the first splits are on their way
// meanwhile, four columns per lane.  With fewer rows than waves the waves of a row share its splits and meet in LDS.
template <int D, int OUT_DT, int WAVES = kMergeWaves>
__device__ __forceinline__ void splitkv_merge_rows(KernargPtr p, char* smem, int b, int h, int row0, int nrows) {
    constexpr int LPR = D / 4, SUBS = 64 / LPR, U = 4;
    const SplitPartials part(p, D, 0);
    const int ns = p->num_splits, lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    int rs_log = 0;                                      // rows side by side: a power of two; G waves share one
    while ((1 << rs_log) < nrows && (1 << rs_log) < WAVES) ++rs_log;
    const int rs = 1 << rs_log, G = WAVES >> rs_log, g = wave >> rs_log;
    const int sub = lane / LPR, col = (lane % LPR) * 4, s_first = g * SUBS + sub, s_step = G * SUBS;
    const uint32_t base = (uint32_t)(b * p->heads + h) * (uint32_t)p->seqlen + (uint32_t)row0;
    if (nrows > WAVES) {
        splitkv_merge_many<D, OUT_DT, WAVES>(p, part, smem, base, p->out + b * p->o_sb + h * p->o_sh + (int64_t)row0 * p->o_sn, nrows, ns, wave, lane);
        return;
    }
    auto row_of = [&](int k) __attribute__((always_inline)) { return (wave & (rs - 1)) + k * rs; };
    auto lse_of = [&](int k) __attribute__((always_inline)) -> float {
        const int r = row_of(k);
        return part.get_lse((uint32_t)(lane < ns ? lane : ns - 1) * part.rows + base + (uint32_t)(r < nrows ? r : nrows - 1));
    };
    auto request = [&](v4f (&x)[U], int k, int s0) __attribute__((always_inline)) {      // s0: a multiple of U * s_step
        const int r = row_of(k);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int s = s0 + u * s_step + s_first;
            if (s0 + u * s_step < ns)                    // (a scalar test; past the end of a last group: any partial, its weight is zero)
                x[u] = part.get((uint32_t)(s < ns ? s : ns - 1) * part.rows + base + (uint32_t)(r < nrows ? r : nrows - 1), D, col);
        }
    };
    char* out0 = p->out + b * p->o_sb + h * p->o_sh + (int64_t)row0 * p->o_sn;
    v4f x[U], x_next[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = x_next[u] = (v4f){0.f, 0.f, 0.f, 0.f};
    float lse = lse_of(0), lse_next = 0.f;
    request(x, 0, 0);
    for (int k = 0; k * rs < nrows; ++k) {
        const bool more = (k + 1) * rs < nrows;
        if (more) {
            lse_next = lse_of(k + 1);
            if (ns <= U * s_step) request(x_next, k + 1, 0);
        }
        lse = lane < ns ? lse : -INFINITY;
        float mx = reduce_wave(lse, [](float a, float c) { return fmaxf(a, c); });
        // A row no split saw a key for: zeros with lse = -inf, as in splitkv_combine_kernel.
        const bool empty = mx == -INFINITY;
        if (empty) mx = 0.f;
        const float total = empty ? -INFINITY : __builtin_log2f(reduce_wave(fast_exp2(lse - mx), [](float a, float c) { return a + c; })) + mx;
        const float w = empty ? 0.f : fast_exp2(lse - total);      // lane s: the weight of split s (0 past the last one)
        const int r = row_of(k);
        if (p->lse != nullptr && g == 0 && lane == 0 && r < nrows) p->lse[base + r] = total;
        v4f acc = {0.f, 0.f, 0.f, 0.f};
        for (int s0 = 0; s0 < ns; s0 += U * s_step) {
            if (s0 != 0) request(x, k, s0);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (s0 + u * s_step >= ns) continue;
                const int s = s0 + u * s_step + s_first;
                const float ws = __shfl(w, s & 63);
                const float wt = s < ns ? ws : 0.f;
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[i] = fmaf(wt, x[u][i], acc[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (SUBS == 4) acc[i] = reduce_row_lanes(acc[i], [](float a, float c) { return a + c; });
            if (SUBS == 2) acc[i] = half_pair_sum(acc[i]);
        }
        if (G > 1) {                                     // (one row per wave then: every wave comes here once)
            v4f* red = (v4f*)(smem + kArrivalBytes);
            static_assert(kArrivalBytes + WAVES * 64 * 16 <= kMergeLds, "");
            if (g > 0) red[wave * 64 + lane] = acc;
            __syncthreads();
            if (g > 0) return;
            for (int j = 1; j < G; ++j) acc += red[(wave + j * rs) * 64 + lane];
        }
        if (sub == 0 && r < nrows) store_out4<OUT_DT>(out0 + (int64_t)r * p->o_sn + col * 2, acc);
        if (more) {
            lse = lse_next;
            if (ns <= U * s_step) {
#pragma unroll
                for (int u = 0; u < U; ++u) x[u] = x_next[u];
            } else {
                request(x, k + 1, 0);
            }
        }
    }
}

// ---- Merge in a launch of its own: D / 4 lanes per output row (one 16-byte load per lane and split, one 8-byte store), 256 / (D / 4) rows per workgroup;
// the loads of four splits are in flight together.
template <int D, int OUT_DT>
__global__ void __launch_bounds__(256) splitkv_combine_kernel(const KParams p) {
    constexpr int LPR = D / 4, RPB = 256 / LPR;
    const int sub = threadIdx.x % LPR, rl = threadIdx.x / LPR;
    const int64_t rows = (int64_t)p.batch * p.heads * p.seqlen;
    const int64_t row = (int64_t)blockIdx.x * RPB + rl;
    if (row >= rows) return;
    const int ns = p.num_splits;
    // log-sum-exp over splits (every lane of a row computes the same scalars)
    float lse_max = -INFINITY;
    for (int s = 0; s < ns; ++s) lse_max = fmaxf(lse_max, p.lse_part[(int64_t)s * rows + row]);
    // A row no split saw a key for (an empty cache entry, a causal row above the first key): every partial is -inf and
    // the result is zeros with lse = -inf, the value the single-pass kernels write for such a row - the neutral element
    // for a caller that merges results by lse.
    const bool empty = lse_max == -INFINITY;
    if (empty) lse_max = 0.f;
    float sum = 0.f;
    for (int s = 0; s < ns; ++s) sum += fast_exp2(p.lse_part[(int64_t)s * rows + row] - lse_max);
    const float lse = empty ? -INFINITY : __builtin_log2f(sum) + lse_max;     // (a NaN partial propagates as NaN)
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    const float* op0 = p.o_part + row * D + sub * 4;
    const int64_t sstride = rows * D;
    for (int s0 = 0; s0 < ns; s0 += 4) {
        v4f part[4];
        float w[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int s = s0 + u < ns ? s0 + u : ns - 1;                 // clamped loads, zero weight past the end
            part[u] = *(const v4f*)(op0 + (int64_t)s * sstride);
            w[u] = (s0 + u < ns && !empty) ? fast_exp2(p.lse_part[(int64_t)s * rows + row] - lse) : 0.f;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] = fmaf(w[u], part[u][i], acc[i]);
    }
    const int64_t bh = row / p.seqlen, n = row % p.seqlen;
    const int64_t b = bh / p.heads, h = bh % p.heads;
    char* orow = p.out + b * p.o_sb + h * p.o_sh + n * p.o_sn + sub * 8;
    store_out4<OUT_DT>(orow, acc);
    if (p.lse != nullptr && sub == 0) p.lse[row] = lse;
}

}  // namespace intfa
