// KV-cache attention for gfx950 (MI355X): in-place append, split-KV partial
// attention over contiguous / remapped / paged caches, log-sum-exp combine.
//
// Replaces csrc/flash_attn/src/kvcache_native.cu: paged_append_kernel
// (:782-871), the contiguous append loop of flash_api.cpp:643-654, the split
// kernels (:148-674) and kvcache_combine_kernel (:676-729).  Semantics kept:
// attention over L = cache_seqlens[b] + seqlen_new keys; split s of S covers
// [L*s/S, L*(s+1)/S) (:191-192); causal keeps key j for query row i iff
// j <= i + L - seqlen_q (:347); GQA kv_head = head / (h/hk) (:341); an empty
// split has LSE -inf and output 0 (:355-372); the combine weights are
// exp(lse_s - lse_total) and a row with no key gets O = 0, LSE = 0 (:697-727);
// probabilities stay fp32 through the PV product (:599, :636-672).
//
// Design: one workgroup per (batch, group of HPI adjacent KV heads, split,
// 32-row tile) where the rows are the q-heads of the GQA group times the query
// positions, so every K/V byte of the split is read once.  The keys of the
// split are walked in 32-key tiles aligned to absolute positions (a tile never
// straddles a page: pages are multiples of 256 tokens); wave w serves head
// w % HPI of the group and its tiles t with t % (4 / HPI) == w / HPI (HPI = 1:
// one head, tile t to wave t % 4).  Each wave
// streams its tiles through a private LDS slot with direct global -> LDS
// copies (global_load_lds): it reads a tile's MFMA operands into registers,
// issues the next tile's copy into the same slot and then computes, so the
// copy is in flight during the compute, with no register staging of the copy
// and no workgroup barrier in the loop.  K stays natural (MFMA A operand
// rows), V natural and read transposed with ds_read_b64_tr_b16.  Each wave
// keeps its own online softmax state; the waves of each head merge their
// partial states through LDS at the end.  Paged, remapped and contiguous
// caches with the same head stride take the same tile order and the same
// arithmetic, so their results are bit-identical for the same logical cache.
// Work items are ordered with the sequence rank slowest: when the caller
// passes a batch_order workspace and there are more items than CUs, one
// workgroup of the append launch first ranks the sequences by key count
// (longest first) and a resident grid of two workgroups per CU deals the items
// out from a device counter in that order, so the longest sequences start
// first, the short ones fill the end, and no workgroup is relaunched between
// items.  With split counts as well, the last split item of each row tile to
// finish combines the tile's partials, so a decode call is two launches.
// Calls of many query rows take kv_chunk_kernel instead (below).
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "fa_common.h"

namespace fa {

constexpr int kKvThreads = 256;
constexpr int kKvWaves = 4;
constexpr int kTile = 32;  // keys per wave tile

__device__ __forceinline__ const f16 *kv_row_ptr(const fa_tensor &t, const fa_kvcache_args &a, int b, int cache_row,
                                                 int hk, int pos) {
    // Element pointer of token `pos` (logical) of sequence b, head hk.
    int64_t off;
    if (a.block_table) {
        const int page = a.page_block_size;
        const int blk = a.block_table[int64_t(b) * a.block_table_stride + pos / page];
        off = int64_t(blk) * t.batch_stride + int64_t(pos % page) * t.row_stride;
    } else {
        off = int64_t(cache_row) * t.batch_stride + int64_t(pos) * t.row_stride;
    }
    return (const f16 *)t.ptr + off + int64_t(hk) * t.head_stride;
}

// Cache length and cache row of sequence b, checked against the cache: a
// negative length, more tokens than the cache holds after the append, or a
// row outside a remapped cache makes the sequence invalid (err bit 1:
// capacity, bit 2: row).  An invalid sequence is not appended to and is
// attended over no keys, so no access leaves the cache whatever the lengths
// and indices hold; the host learns of it from the status word.
struct KvSeq {
    int L0;   // tokens in the cache before the append (0 when invalid)
    int row;  // cache row (contiguous cache)
    int err;
};
__device__ __forceinline__ KvSeq kv_seq(const fa_kvcache_args &a, int b) {
    KvSeq s;
    s.L0 = a.cache_seqlens[b];
    s.row = a.cache_batch_idx ? a.cache_batch_idx[b] : b;
    s.err = (s.L0 < 0 || (a.cache_capacity > 0 && int64_t(s.L0) + a.seqlen_new > a.cache_capacity) ? 1 : 0) |
            (a.cache_batch_idx && a.cache_batch > 0 && (s.row < 0 || s.row >= a.cache_batch) ? 2 : 0);
    if (s.err) {
        s.L0 = 0;
        s.row = 0;
    }
    return s;
}

// Rotary embedding of the 8 channels [c0, c0 + 8) of one row (c0 a multiple of
// 8 below rotary_dim) at position pos: x holds them, row points at channel 0
// of the row (the non-interleaved form reads the partner channels there).
// Each output is x_a * cos - x_b * sin or x_a * sin + x_b * cos in fp32; the
// products of fp16 values are exact in fp32, so it is the exact rotation of
// the fp16 inputs rounded once to fp32, then to fp16.
typedef f16 f16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x4 rotary8(const fa_kvcache_args &a, const u32x4 x, const f16 *row, int c0, int pos) {
    // Opaque to the optimiser: keeps the per-channel table addresses from being
    // hoisted out of the split kernel's item loop, where they would stay live
    // (in spilled registers) through it.
    asm volatile("" : "+v"(c0));
    const int half = a.rotary_dim / 2;
    const int64_t base = int64_t(min(max(pos, 0), a.rotary_seqlen - 1)) * half;
    const f16 *cs = (const f16 *)a.rotary_cos + base;
    const f16 *sn = (const f16 *)a.rotary_sin + base;
    const f16x8 xv = as_h8(x);
    f16x8 r;
    if (a.rotary_interleaved) {
        const f16x4 c = *reinterpret_cast<const f16x4 *>(cs + c0 / 2);
        const f16x4 s = *reinterpret_cast<const f16x4 *>(sn + c0 / 2);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float x0 = float(xv[2 * e]), x1 = float(xv[2 * e + 1]);
            const float ce = float(c[e]), se = float(s[e]);
            r[2 * e] = f16(x0 * ce - x1 * se);
            r[2 * e + 1] = f16(x0 * se + x1 * ce);
        }
    } else {
        const bool first = c0 < half;
        const int j0 = first ? c0 : c0 - half;
        const f16x8 pv = as_h8(ldg16(row + (first ? c0 + half : j0)));
        const f16x8 c = as_h8(ldg16(cs + j0));
        const f16x8 s = as_h8(ldg16(sn + j0));
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float xe = float(xv[e]), pe = float(pv[e]), ce = float(c[e]), se = float(s[e]);
            r[e] = f16(first ? xe * ce - pe * se : xe * ce + pe * se);
        }
    }
    return __builtin_bit_cast(u32x4, r);
}

// ---------------------------------------------------------------------------
// Append of 16-byte chunk idx of k_new / v_new, one per thread (with
// rotary_dim > 0, the key chunks below rotary_dim are rotated at their
// position first).
template <int HD>
__device__ __forceinline__ void append_chunk(const fa_kvcache_args &a, const int64_t idx) {
    constexpr int KCH = HD / 8;
    const int64_t total = int64_t(a.batch) * a.seqlen_new * a.nheads_k * KCH;
    if (idx >= total) return;
    const int c = int(idx % KCH);
    int64_t rest = idx / KCH;
    const int hk = int(rest % a.nheads_k);
    rest /= a.nheads_k;
    const int t = int(rest % a.seqlen_new);
    const int b = int(rest / a.seqlen_new);
    const KvSeq sq = kv_seq(a, b);
    if (sq.err) {
        if (a.status && idx % (int64_t(a.seqlen_new) * a.nheads_k * KCH) == 0) atomicOr(a.status, sq.err);
        return;
    }
    const int pos = sq.L0 + t;
    const int cache_row = sq.row;
    const f16 *ks = (const f16 *)a.k_new.ptr + int64_t(b) * a.k_new.batch_stride + int64_t(t) * a.k_new.row_stride +
                    int64_t(hk) * a.k_new.head_stride + 8 * c;
    const f16 *vs = (const f16 *)a.v_new.ptr + int64_t(b) * a.v_new.batch_stride + int64_t(t) * a.v_new.row_stride +
                    int64_t(hk) * a.v_new.head_stride + 8 * c;
    f16 *kd = const_cast<f16 *>(kv_row_ptr(a.k_cache, a, b, cache_row, hk, pos)) + 8 * c;
    f16 *vd = const_cast<f16 *>(kv_row_ptr(a.v_cache, a, b, cache_row, hk, pos)) + 8 * c;
    u32x4 kx = ldg16(ks);
    if (8 * c < a.rotary_dim) kx = rotary8(a, kx, ks - 8 * c, 8 * c, pos);
    *reinterpret_cast<u32x4 *>(kd) = kx;
    *reinterpret_cast<u32x4 *>(vd) = ldg16(vs);
}

// ---------------------------------------------------------------------------
// Append and ordering in one launch of kOrderThreads-thread workgroups.  The
// first order_wgs workgroups (0 or 1) rank the sequences: batch_order[r] = the
// sequence with the r-th most keys, by a counting sort over key-count buckets
// (exact below 32 keys, then 32 buckets per power of two: about 3 % apart;
// order within a bucket is arbitrary, which changes no result), and zero the
// split kernel's work counter batch_order[batch] and its n_count split counts
// (the counts alone without rank).
// The other workgroups append one 16-byte chunk per thread.  The two parts
// touch disjoint memory (the ranking reads cache_seqlens only).
__device__ __forceinline__ int kv_len_bucket(int n) {
    if (n < 32) return n;
    const int msb = 31 - __clz(n);
    return (msb - 4) * 32 + ((n >> (msb - 5)) & 31);
}
template <int HD>
__global__ __launch_bounds__(kOrderThreads) void kv_prep_kernel(const fa_kvcache_args a, const int order_wgs,
                                                                const bool rank, int32_t *const count,
                                                                const int n_count) {
    if (int(blockIdx.x) < order_wgs) {
        for (int i = threadIdx.x; i < n_count; i += kOrderThreads) count[i] = 0;
        if (!rank) return;
        if (threadIdx.x == 0) a.batch_order[a.batch] = 0;
        order_items(
            a.batch,
            [&](int b) {
                const KvSeq sq = kv_seq(a, b);
                return kv_len_bucket(sq.err ? 0 : sq.L0 + a.seqlen_new);
            },
            a.batch_order, true);
        return;
    }
    append_chunk<HD>(a, int64_t(blockIdx.x - order_wgs) * kOrderThreads + threadIdx.x);
}

// ---------------------------------------------------------------------------
// Combine of NR output rows r[] (of batch * nheads * seqlen_q) by one wave.  Lane
// s reads split s's LSE of every row (further rounds past 64 splits) while the
// partial outputs of the first PRE splits of all rows are loaded at the same
// time, so the rows share one round trip to memory; the maximum and the weight
// sum are wave reductions, and each lane sums HD / 64 output elements over the
// splits with the weight exp(lse_s - lse_total) taken from lane s.  Run by the
// combine kernel, or inside the split kernel by the last split item of a row
// tile.  n: rows that count (the others repeat one, and are not stored).
constexpr int kPreSplits = 16;

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v = fmaxf(v, __shfl_xor(v, m));
    return v;
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m);
    return v;
}

// Split partials as the combine reads them.  Inside the split kernel
// (COHERENT) they are device-scope atomic loads, which see what device-scope
// stores of other workgroups left whatever this XCD's L2 holds (the partials
// are stored that way); the combine kernel, launched after the split kernel,
// reads them plainly.
template <bool COHERENT>
__device__ __forceinline__ float load_part(const float *p) {
    if constexpr (COHERENT)
        return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
        return *p;
}
template <bool COHERENT, int DPL>
__device__ __forceinline__ float __attribute__((ext_vector_type(DPL))) load_part_vec(const float *p) {
    typedef float fdpl __attribute__((ext_vector_type(DPL)));
    if constexpr (!COHERENT) {
        return *reinterpret_cast<const fdpl *>(p);
    } else if constexpr (DPL == 1) {
        fdpl v;
        v[0] = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return v;
    } else {
        static_assert(DPL == 2, "one 64-bit load per lane");
        const uint64_t u =
            __hip_atomic_load(reinterpret_cast<const uint64_t *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return __builtin_bit_cast(fdpl, u);
    }
}

template <int HD, bool COHERENT, int NR, int PRE>
__device__ __forceinline__ void combine_rows(const fa_kvcache_args &a, const int (&r)[NR], int n, int lane) {
    // Opaque to the optimiser: keeps the addresses below from being hoisted out
    // of the split kernel's item loop into registers live through its tile loop.
    asm volatile("" : "+v"(lane));
    constexpr int DPL = HD / 64;  // output elements per lane
    typedef float fdpl __attribute__((ext_vector_type(DPL)));
    const int nrow = a.batch * a.nheads * a.seqlen_q;
    const int S = a.num_splits;
    auto part = [&](int s, int row) {
        return load_part_vec<COHERENT, DPL>(a.out_accum + (int64_t(s) * nrow + row) * HD + DPL * lane);
    };
    auto lse_of = [&](int s, int row) { return load_part<COHERENT>(a.lse_accum + int64_t(s) * nrow + row); };
    // Splits past S re-read split S - 1 (finite) and get weight 0 below.
    fdpl pre[NR][PRE];
    float lse0[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
#pragma unroll
        for (int s = 0; s < PRE; ++s) pre[i][s] = part(min(s, S - 1), r[i]);
        lse0[i] = lane < S ? lse_of(lane, r[i]) : -INFINITY;
    }
#pragma unroll
    for (int i = 0; i < NR; ++i) {
        float lmax = lse0[i];
        for (int s0 = 64; s0 < S; s0 += 64)
            if (s0 + lane < S) lmax = fmaxf(lmax, lse_of(s0 + lane, r[i]));
        lmax = wave_max(lmax);
        float psum = 0.f;
        if (lmax != -INFINITY) {
            if (lane < S) psum = expf(lse0[i] - lmax);
            for (int s0 = 64; s0 < S; s0 += 64)
                if (s0 + lane < S) psum += expf(lse_of(s0 + lane, r[i]) - lmax);
        }
        const float wsum = wave_sum(psum);
        const bool live = lmax != -INFINITY && wsum > 0.f;
        const float ltot = live ? lmax + logf(wsum) : -INFINITY;
        fdpl acc;
#pragma unroll
        for (int e = 0; e < DPL; ++e) acc[e] = 0.f;
        if (live) {
            const float w0 = lane < S ? expf(lse0[i] - ltot) : 0.f;
            auto weight = [](float w, int s) {
                return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w), s));
            };
#pragma unroll
            for (int s = 0; s < PRE; ++s) acc += weight(w0, s) * pre[i][s];  // lane s >= S holds w0 = 0
            for (int s0 = 0; s0 < S; s0 += 64) {
                const float w = s0 == 0 ? w0 : (s0 + lane < S ? expf(lse_of(s0 + lane, r[i]) - ltot) : 0.f);
                const int m = min(64, S - s0);
#pragma unroll 1
                for (int s = s0 == 0 ? PRE : 0; s < m; ++s) acc += weight(w, s) * part(s0 + s, r[i]);
            }
        }
        if (i < n) {
            const int qp = r[i] % a.seqlen_q;
            const int bh = r[i] / a.seqlen_q;
            const int h = bh % a.nheads, b = bh / a.nheads;
            f16 *op = (f16 *)a.o.ptr + int64_t(b) * a.o.batch_stride + int64_t(qp) * a.o.row_stride +
                      int64_t(h) * a.o.head_stride + DPL * lane;
#pragma unroll
            for (int e = 0; e < DPL; ++e) op[e] = (f16)acc[e];
            if (lane == 0) a.lse[r[i]] = live ? ltot : 0.f;
        }
    }
}

// ---------------------------------------------------------------------------
// Split-KV partial attention.
template <int HD>
struct KvCfg {
    static constexpr int KCH = HD / 8;
    static constexpr int TILE = kTile * HD * 2;         // one K or V tile, natural layout
    static constexpr int STAGE = 2 * TILE;              // K tile, then V tile
    // Ring stages per wave.  A tile's operands are read into registers and the
    // stage is refilled before the tile is computed, so one stage keeps a tile
    // in flight; at head_dim 64 a second stage (more bytes in flight, +1 % on a
    // long-context decode) still lets two workgroups share a CU, at 128 it
    // would not (one's start-up and merge overlap the other's streaming).
    static constexpr int NST = HD == 64 ? 2 : 1;
    // Also holds HD x 32 fp32 at the merge, at a row stride of 33: a row's
    // dimensions, which neighbouring lanes read, then lie in different banks.
    static constexpr int MERGE = 33;
    static constexpr int WAVE_LDS = NST * STAGE > HD * MERGE * 4 ? NST * STAGE : HD * MERGE * 4;
    static_assert(WAVE_LDS % 512 == 0, "tile bases must be multiples of 512 bytes");
    static constexpr int CPW = kTile * KCH / 64;        // copies per lane per tile (K or V)
    static constexpr int MAX_PAGES = 1024;              // page ids of one split staged in LDS
};

// The running maximum m that a row's probabilities P = exp2(S*c - m) are taken
// against is raised (and O, l rescaled) only when some row of the wave finds a
// score more than this many doublings above it; P stays below 2^8, and its hi +
// lo fp16 halves still carry about 22 bits.
constexpr float kKvRescaleSlack = 8.f;

// tanh x = 1 - 2 / (e^(2x) + 1): exactly +-1 at the ends, an absolute error of a
// few fp32 ulps of 1 in between (what a softcapped score needs).
__device__ __forceinline__ float tanh_fast(float x) {
    const float e = exp2_fast(x * (2.f * kLog2e));
    return 1.f - 2.f * __builtin_amdgcn_rcpf(e + 1.f);
}

// Work items are (sequence rank, split, kv head, row tile), rank slowest: with
// batch_order the longest sequences' items come first (longest-job-first keeps
// the last items short).  With DYN the grid is resident (two workgroups per
// CU) and each workgroup, after its first item blockIdx.x, takes the next
// unclaimed item from a device counter, so no workgroup is relaunched and
// the items are dealt out greedily in that order.  The counter
// (batch_order[batch]) is zeroed by kv_prep_kernel on the same stream; an item
// that finds the whole list under way claims nothing.  With at most one item
// per CU the sequences are taken as they come (ranked is false) and not ranked:
// one sequence of 1500 tokens, 32 / 8 heads, 17.8 -> 15.7 us a call.  With two
// per CU the order still pairs long items with short ones (64 sequences of 1.5k
// - 3k tokens, 512 items: 117 us ranked, 122 not).
// With count (num_splits > 1, DYN) the split kernel also combines: count[(b *
// nheads_k + hk) * row_tiles + rt] (zeroed by kv_prep_kernel) counts the
// finished splits of that row tile, and the item that finishes last combines
// the tile's rows with combine_rows, as the combine kernel would.
// EXT switches on the local window, softcap, ALiBi, cache_leftpad and rotary options
// (a separate instance, so the plain kernel carries none of their work).
// HPI (1, 2 or 4) KV heads per item: wave w serves head hk0 + w % HPI and
// takes every (4 / HPI)-th tile of it, so at one key position the waves of a
// workgroup read HPI adjacent heads' rows, HPI * head_dim * 2 contiguous bytes
// of a head-interleaved cache row, where one head alone reads 128 or 256.
template <int HD, bool DYN, bool EXT, int HPI>
__global__ __launch_bounds__(256, 2) void kv_splitkv_kernel(const fa_kvcache_args a, const int row_tiles,
                                                            const int n_items, int32_t *const count,
                                                            const bool ranked) {
    using C = KvCfg<HD>;
    static_assert(HPI == 1 || HPI == 2 || HPI == 4, "heads per item");
    constexpr int WPH = kKvWaves / HPI;  // waves per head
    __shared__ __attribute__((aligned(16))) char smem[kKvWaves * C::WAVE_LDS + kKvWaves * 2 * 32 * 4];
    __shared__ int pages[C::MAX_PAGES];
    __shared__ int next_item, last_item;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: scalar loop control
    const int col = lane & 31, hh = lane >> 5;
    const int n_groups = a.nheads_k / HPI;
    for (int item = blockIdx.x; item < n_items;) {
        int rest = item;
        const int rt = rest % row_tiles;
        rest /= row_tiles;
        const int hk0 = (rest % n_groups) * HPI;  // the item's first KV head
        const int hk = hk0 + wave % HPI;          // this wave's
        rest /= n_groups;
        const int split = rest % a.num_splits;
        const int rank = rest / a.num_splits;
        const int b = DYN && ranked ? a.batch_order[rank] : rank;
        const int G = a.nheads / a.nheads_k;
        const int R = G * a.seqlen_q;  // rows of this (batch, kv head): row = qpos * G + g

        const KvSeq sq = kv_seq(a, b);
        if (sq.err && a.status && tid == 0) atomicOr(a.status, sq.err);
        const int L = sq.err ? 0 : sq.L0 + a.seqlen_new;
        const int S = a.num_splits;
        // Valid keys [kstart, kend): cache_leftpad moves the start (positions
        // stay), and a local window leaves those that some row of the tile sees,
        // so that every split has its share of what is read (16 sequences of 512
        // - 8192 tokens, 4096-key window, 2 splits: 83 -> 64 us a call against
        // splits of the whole sequence, some of them outside the window).
        int kstart = EXT && a.cache_leftpad ? min(max(a.cache_leftpad[b], 0), L) : 0, kend = L;
        const int p_first = (rt * 32) / G + L - a.seqlen_q;                   // key positions of the tile's
        const int p_last = (min(R, rt * 32 + 32) - 1) / G + L - a.seqlen_q;  // first and last query
        if constexpr (EXT) {
            if (a.local_window) {
                if (a.window_left >= 0) kstart = max(kstart, p_first - a.window_left);
                if (a.causal) kend = min(kend, p_last + 1);
                if (a.window_right >= 0) kend = min(kend, p_last + a.window_right + 1);
                kend = max(kend, kstart);
            }
        }
        const int s0 = kstart + int((int64_t(kend - kstart) * split) / S);
        const int s1 = kstart + int((int64_t(kend - kstart) * (split + 1)) / S);
        const int cache_row = sq.row;

        // This lane's query row.
        const int row = rt * 32 + col;
        const bool row_ok = row < R;
        const int qpos = row_ok ? row / G : 0;
        const int hq = hk * G + (row_ok ? row % G : 0);
        int lim = a.causal ? qpos + L - a.seqlen_q : L - 1;  // last visible key
        int w_lo = 0;                                          // first visible key
        // Wave-uniform bounds of the keys every row of the tile sees: tiles in
        // [max(s0, wlo_max), min(s1, lim_min + 1)) need no mask.
        int lim_min = a.causal ? p_first : L - 1;
        int wlo_max = 0;
        if constexpr (EXT) {
            if (a.local_window) {
                const int pos = qpos + L - a.seqlen_q;  // the query's own key position
                if (a.window_right >= 0) {
                    lim = min(lim, pos + a.window_right);
                    lim_min = min(lim_min, p_first + a.window_right);
                }
                if (a.window_left >= 0) {
                    w_lo = pos - a.window_left;
                    wlo_max = p_last - a.window_left;
                }
            }
        }

        const bool neg = a.softmax_scale < 0.f;
        const bool capped = EXT && a.softcap > 0.f;
        const bool alibi = EXT && a.alibi_slopes != nullptr;
        // Softcapped or biased scores are formed in natural units (scaled), so
        // the exponent multiplier is log2(e) for them and scale * log2(e)
        // otherwise; cap_in = scale / softcap.
        const bool natural = capped || alibi;
        const float cscale = natural ? kLog2e : fabsf(a.softmax_scale) * kLog2e;
        const float cap_in = capped ? fabsf(a.softmax_scale) / a.softcap : 0.f;
        const float slope = alibi ? a.alibi_slopes[int64_t(b) * a.alibi_batch_stride + hq] : 0.f;
        const int qkey = qpos + L - a.seqlen_q;  // the query's own key position (ALiBi distance origin)
        // Rotary position of the query: its own (cache_seqlens + i) when causal
        // or windowed, else cache_seqlens for every row.
        const int rpos = sq.L0 + (a.causal || a.local_window ? qpos : 0);
        f16x8 qB[HD / 16];
        {
            const f16 *qp = (const f16 *)a.q.ptr + int64_t(b) * a.q.batch_stride + int64_t(qpos) * a.q.row_stride +
                            int64_t(hq) * a.q.head_stride;
    #pragma unroll
            for (int g = 0; g < HD / 16; ++g) {
                u32x4 v = row_ok ? ldg16(qp + 16 * g + 8 * hh) : zero_u4();
                if (EXT && row_ok && 16 * g + 8 * hh < a.rotary_dim) v = rotary8(a, v, qp, 16 * g + 8 * hh, rpos);
                if (neg) v = neg_h8(v);
                qB[g] = as_h8(v);
            }
        }

        f32x16 o[HD / 32];
    #pragma unroll
        for (int i = 0; i < HD / 32; ++i) o[i] = zero16();
        float m_t = -INFINITY, l_p = 0.f;

        const int t_first = s0 / kTile;
        const int t_last = s1 > s0 ? (s1 - 1) / kTile : t_first - 1;
        const int my_first = t_first + wave / HPI;
        const int n_my = my_first <= t_last ? (t_last - my_first) / WPH + 1 : 0;

        // Page ids of the split, staged in LDS so the ring never waits on a table read.
        const int page = a.page_block_size;
        const int pg_first = a.block_table ? (t_first * kTile) / page : 0;
        const int n_pages = a.block_table && s1 > s0 ? (t_last * kTile) / page - pg_first + 1 : 0;
        const bool pages_in_lds = n_pages <= C::MAX_PAGES;
        if (a.block_table && pages_in_lds) {
            const int32_t *bt = a.block_table + int64_t(b) * a.block_table_stride + pg_first;
            // Opaque start index: keeps this loop's per-lane addresses from being
            // hoisted out of the item loop (and spilled in the options instance).
            int i0 = tid;
            asm volatile("" : "+v"(i0));
            for (int i = i0; i < n_pages; i += kKvThreads) pages[i] = bt[i];
        }
        __syncthreads();

        const int64_t krs = a.k_cache.row_stride, vrs = a.v_cache.row_stride;

        // The tile loop, instantiated twice: with the split's page ids in LDS (and
        // no other vector-memory load while copies are in flight), and a fallback
        // that reads the block table per tile for splits spanning more pages.
        auto run = [&](auto lds_pages_tag) {
        constexpr bool LDS_PAGES = decltype(lds_pages_tag)::value;
        // Copy tile t into ring stage st of this wave.  Rows past L re-read key L - 1
        // of the same tile (finite values; masked below).
        auto issue = [&](int t, int st) {
            const int p0 = t * kTile;
            int64_t koff, voff;
            if (a.block_table) {
                const int pi = p0 / page;
                int blk;
                if constexpr (LDS_PAGES)
                    blk = pages[pi - pg_first];
                else
                    blk = a.block_table[int64_t(b) * a.block_table_stride + pi];
                const int in_page = p0 - pi * page;
                koff = int64_t(blk) * a.k_cache.batch_stride + int64_t(in_page) * krs;
                voff = int64_t(blk) * a.v_cache.batch_stride + int64_t(in_page) * vrs;
            } else {
                koff = int64_t(cache_row) * a.k_cache.batch_stride + int64_t(p0) * krs;
                voff = int64_t(cache_row) * a.v_cache.batch_stride + int64_t(p0) * vrs;
            }
            const f16 *kb = (const f16 *)a.k_cache.ptr + koff + int64_t(hk) * a.k_cache.head_stride;
            const f16 *vb = (const f16 *)a.v_cache.ptr + voff + int64_t(hk) * a.v_cache.head_stride;
            char *ks = smem + wave * C::WAVE_LDS + st * C::STAGE;
            char *vs = ks + C::TILE;
            dma_tile<HD, kTile, 64>(ks, kb, krs, 0, L - 1 - p0, 0, lane);
            dma_tile<HD, kTile, 64>(vs, vb, vrs, 0, L - 1 - p0, 0, lane);
        };

        TileReader<HD> rd;
        rd.init(lane);
        if (n_my > 0) issue(my_first, 0);
        if (C::NST > 1 && n_my > 1) issue(my_first + WPH, 1);
        for (int k = 0; k < n_my; ++k) {
            const int st = k % C::NST;
            if (k + 1 < n_my)
                wait_vmem_n<(C::NST - 1) * 2 * C::CPW>();  // newer tiles may stay in flight
            else
                wait_vmem();
            const char *ks = smem + wave * C::WAVE_LDS + st * C::STAGE;
            const char *vs = ks + C::TILE;
            const int p0 = (my_first + k * WPH) * kTile;
            // All operands of the tile into registers first, then refill the stage
            // right away: two tiles stay in flight while this one is computed.
            f16x8 ka[HD / 16], va[HD / 32][2];
    #pragma unroll
            for (int g = 0; g < HD / 16; ++g) ka[g] = rd.a_operand(ks, 0, g);
    #pragma unroll
            for (int dt = 0; dt < HD / 32; ++dt)
    #pragma unroll
                for (int gg = 0; gg < 2; ++gg) va[dt][gg] = rd.tr_operand(vs, 16 * gg, dt);
            wait_lds();
            if (k + C::NST < n_my) issue(my_first + (k + C::NST) * WPH, st);
            f32x16 s = mfma32(ka[0], qB[0], zero16());
    #pragma unroll
            for (int g = 1; g < HD / 16; ++g) s = mfma32(ka[g], qB[g], s);
            if constexpr (EXT) {
                if (natural) {
                    const float sc = fabsf(a.softmax_scale);
    #pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        float x = capped ? a.softcap * tanh_fast(s[r] * cap_in) : s[r] * sc;
                        if (alibi) x -= slope * float(abs(qkey - (p0 + acc_lrow(r, hh))));
                        s[r] = x;
                    }
                }
            }
            float mx = -INFINITY;
            const bool interior = p0 >= s0 && p0 + kTile <= s1 && p0 + kTile - 1 <= lim_min && p0 >= wlo_max;
            if (interior) {
    #pragma unroll
                for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
            } else {
    #pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int key = p0 + acc_lrow(r, hh);
                    if (key < s0 || key >= s1 || key > lim || (EXT && key < w_lo)) s[r] = -INFINITY;
                    mx = fmaxf(mx, s[r]);
                }
            }
            mx = max_xor32(mx);
            const float mx_t = mx == -INFINITY ? -INFINITY : mx * cscale;
            if (__builtin_amdgcn_ballot_w64(mx_t > m_t + kKvRescaleSlack) != 0) {
                const float m_new = fmaxf(m_t, mx_t);
                const float alpha = m_new == -INFINITY ? 1.f : exp2_fast(m_t - m_new);
                l_p *= alpha;
    #pragma unroll
                for (int dt = 0; dt < HD / 32; ++dt)
    #pragma unroll
                    for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
                m_t = m_new;
            }
            const float m_use = m_t == -INFINITY ? 0.f : m_t;
            // A masked score is -inf after every transform, and exp2(-inf) = 0.
            float rs = 0.f;
    #pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float p = exp2_fast(fmaf(s[r], cscale, -m_use));
                s[r] = p;
                rs += p;
            }
            l_p += rs;
            // P stays fp32-accurate through the product: P = hi + lo with both halves fp16.
            f16x8 ph[2], pl[2];
    #pragma unroll
            for (int gg = 0; gg < 2; ++gg)
    #pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const float p = s[8 * gg + u];
                    const f16 hi = (f16)p;
                    ph[gg][u] = hi;
                    pl[gg][u] = (f16)(p - float(hi));
                }
    #pragma unroll
            for (int dt = 0; dt < HD / 32; ++dt) {
    #pragma unroll
                for (int gg = 0; gg < 2; ++gg) {
                    o[dt] = mfma32(va[dt][gg], ph[gg], o[dt]);
                    o[dt] = mfma32(va[dt][gg], pl[gg], o[dt]);
                }
            }
        }
        };
        if (pages_in_lds)
            run(std::true_type{});
        else
            run(std::false_type{});

        // Merge the waves of each head (waves j, j + HPI, ...): each publishes
        // (m, l) per row and its O^T tile.
        const float l_w = sum_xor32(l_p);
        float *mrow = reinterpret_cast<float *>(smem + kKvWaves * C::WAVE_LDS);
        float *lrow = mrow + kKvWaves * 32;
        __syncthreads();  // every wave is done with its ring
        float *ow = reinterpret_cast<float *>(smem + wave * C::WAVE_LDS);  // [HD][MERGE] fp32
    #pragma unroll
        for (int dt = 0; dt < HD / 32; ++dt)
    #pragma unroll
            for (int r = 0; r < 16; ++r) ow[(dt * 32 + acc_row(r, hh)) * C::MERGE + col] = o[dt][r];
        if (hh == 0) {
            mrow[wave * 32 + col] = m_t;
            lrow[wave * 32 + col] = l_w;
        }
        __syncthreads();

        const int rows_here = min(32, R - rt * 32);
        const int nrow_all = a.batch * a.nheads * a.seqlen_q;
        for (int e = tid; e < HPI * rows_here * HD; e += kKvThreads) {
            const int j = e / (rows_here * HD), c = (e / HD) % rows_here, d = e % HD;
            float mstar = -INFINITY;
    #pragma unroll
            for (int i = 0; i < WPH; ++i) mstar = fmaxf(mstar, mrow[(j + HPI * i) * 32 + c]);
            float lsum = 0.f, acc = 0.f;
            if (mstar != -INFINITY) {
    #pragma unroll
                for (int i = 0; i < WPH; ++i) {
                    const int w = j + HPI * i;
                    const float mw = mrow[w * 32 + c];
                    const float sc = mw == -INFINITY ? 0.f : exp2_fast(mw - mstar);
                    lsum += lrow[w * 32 + c] * sc;
                    acc += reinterpret_cast<const float *>(smem + w * C::WAVE_LDS)[d * C::MERGE + c] * sc;
                }
            }
            const bool live = lsum > 0.f;
            const float outv = live ? acc / lsum : 0.f;
            const float lse = live ? (mstar + log2_fast(lsum)) * kLn2 : -INFINITY;
            const int r = rt * 32 + c;
            const int qp = r / G, h = (hk0 + j) * G + r % G;
            const int64_t orow = (int64_t(b) * a.nheads + h) * a.seqlen_q + qp;  // (batch, head, qpos)
            if (S == 1) {
                f16 *op = (f16 *)a.o.ptr + int64_t(b) * a.o.batch_stride + int64_t(qp) * a.o.row_stride +
                          int64_t(h) * a.o.head_stride;
                op[d] = (f16)outv;
                if (d == 0) a.lse[orow] = live ? lse : 0.f;
            } else {
                // Device-scope stores: the last split item of the tile may combine
                // them on another XCD in this same launch.
                __hip_atomic_store(a.out_accum + (int64_t(split) * nrow_all + orow) * HD + d, outv, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
                if (d == 0)
                    __hip_atomic_store(a.lse_accum + int64_t(split) * nrow_all + orow, lse, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        if (DYN && S > 1 && count) {
            // The item counts itself done once every wave's partial stores have
            // completed (vmcnt 0: written at device scope); the item that brings
            // the count to S has seen all S items' stores complete and reads the
            // partials with device-scope loads.  No cache-wide write-back or
            // invalidate is needed (both would stall this XCD's L2 once per item).
            // This rests on gfx950's agent-scope accesses, not on the HIP memory
            // model (the atomics are relaxed): an agent-scope store is written
            // past the XCD's L2 before its vmcnt completes, and an agent-scope
            // load does not hit another XCD's stale L2 copy; the #error at the
            // top of fa_common.h keeps other targets from building it.  The count
            // of a row tile of a head group sits at its first head's slot.
            wait_vmem();
            __syncthreads();
            if (tid == 0)
                last_item = __hip_atomic_fetch_add(count + (int64_t(b) * a.nheads_k + hk0) * row_tiles + rt, 1,
                                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == S - 1;
            __syncthreads();
            if (last_item) {
                // Up to 4 rows at a time and wave: one by one, each waited a round trip
                // to memory (16 rows in 16 splits: 28.7 -> 25.3 us a call, 32: 43 -> 37).
                const int n_rows = HPI * rows_here;
                auto rows = [&](auto nr_tag, auto pre_tag) FA_INLINE {
                    constexpr int NR = decltype(nr_tag)::value;
                    for (int c = wave; c < n_rows; c += NR * kKvWaves) {
                        int r[NR];
#pragma unroll
                        for (int i = 0; i < NR; ++i) {
                            const int x = min(c + i * kKvWaves, n_rows - 1), j = x / rows_here;
                            const int row = rt * 32 + x - j * rows_here;
                            r[i] = (b * a.nheads + (hk0 + j) * G + row % G) * a.seqlen_q + row / G;
                        }
                        combine_rows<HD, true, NR, decltype(pre_tag)::value>(a, r, (n_rows - 1 - c) / kKvWaves + 1, lane);
                    }
                };
                using Pre = std::integral_constant<int, kPreSplits>;
                using I1 = std::integral_constant<int, 1>;
                using I2 = std::integral_constant<int, 2>;
                using I4 = std::integral_constant<int, 4>;
                if (n_rows <= kKvWaves)
                    rows(I1{}, Pre{});
                else if (n_rows <= 2 * kKvWaves)
                    rows(I2{}, Pre{});
                else if (S <= 4)
                    rows(I4{}, I4{});
                else
                    rows(I4{}, Pre{});
            }
        }
        if (!DYN || n_items <= int(gridDim.x)) break;
        __syncthreads();  // every thread is done with this item's LDS
        if (tid == 0) next_item = atomicAdd(a.batch_order + a.batch, 1) + int(gridDim.x);
        __syncthreads();
        item = next_item;
    }
}

// ---------------------------------------------------------------------------
// Many query rows per KV head (prompt chunks).  kv_splitkv_kernel reads a
// split's K / V once per 32 rows, each wave its own tiles: at 512 tokens x 4
// heads it reads them 64 times and runs at the L2's rate.  Here a workgroup
// holds 128 rows, 32 per wave, and its waves share every 64-key block through
// LDS (two stages, one barrier a block, two workgroups per CU), as in the
// forward kernel; P still goes through PV as hi + lo fp16 halves, so each V
// operand read from LDS feeds two MFMAs, and the matrix cores bound it (48
// MFMAs a 32 x 64 block and wave against 326 VALU instructions).  Two sequences
// of 512 tokens on 4k - 12k keys, 32 / 8 heads, head_dim 128: 452 -> 205 us a
// call (288 -> 635 TFLOP/s with PV counted once, about 950 as executed).
// Items, their order and the options are kv_splitkv_kernel's; a split takes a
// share of the keys that some row of its tile sees (with a window those are
// few of the sequence's).  With num_splits > 1 the last split of a row tile to
// finish adds the others' partials to its own.
constexpr int kChunkRows = 128, kChunkKeys = 64;
// Page ids in LDS: as many as fit beside the stages of two workgroups per CU (about
// a million tokens in pages of 256).  Staging them anew on the way, for any number,
// cost the block loop 0.6 - 1.2 % (two sequences of 512 tokens: 215 -> 217.6 us).
constexpr int kChunkPages = 3840;
constexpr int kChunkMinRows = 64, kChunkMaxSplits = 32;

// Merges the partial rows (O normalised, LSE) of a row tile's splits.  Every
// item stores its own, lane by lane, and then counts itself; the one that
// counts last, or that finds all others counted before it has stored anything,
// sums them in split order, its own from registers, so no item waits for another.  row0: the tile's first row of
// a split's accumulators, rows_here x HD values from there.  Returns whether
// this item holds the sum.
template <int HD>
__device__ __forceinline__ bool chunk_merge(const fa_kvcache_args &a, int32_t *count, int split, int64_t row0,
                                            int rows_here, int row, int hh, int *ticket, f32x16 (&o)[HD / 32],
                                            float &lse) {
    constexpr int N = HD / 4;  // pairs of floats a lane holds
    const int S = a.num_splits, tid = threadIdx.x;
    const int64_t nrow = int64_t(a.batch) * a.nheads * a.seqlen_q;
    const bool live = row < rows_here;
    // Pair i of a lane: element (2 i + hh) * rows_here + row, 256 contiguous bytes a half wave.
    uint64_t *pairs = reinterpret_cast<uint64_t *>(a.out_accum + row0 * HD) + hh * rows_here + row;
    const int step = 2 * rows_here;
    float *lses = a.lse_accum + row0 + row;
    if (tid == 0) *ticket = __hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*ticket != S - 1) {
        if (live) {
            uint64_t *slot = pairs + int64_t(split) * nrow * (HD / 2);
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const f32x2 x = {o[i / 8][2 * (i & 7)], o[i / 8][2 * (i & 7) + 1]};
                __hip_atomic_store(slot + i * step, __builtin_bit_cast(uint64_t, x), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            }
            if (hh == 0)
                __hip_atomic_store(lses + int64_t(split) * nrow, lse, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        wait_vmem();
        __syncthreads();  // every wave's stores have completed
        if (tid == 0) *ticket = __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (*ticket != S - 1) return false;
    }
    if (!live) return true;
    auto lse_of = [&](int s) {
        return s == split ? lse
                          : __hip_atomic_load(lses + int64_t(s) * nrow, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    float mx = -INFINITY, sum = 0.f;
    for (int s = 0; s < S; ++s) mx = fmaxf(mx, lse_of(s));
    for (int s = 0; s < S; ++s) sum += mx == -INFINITY ? 0.f : expf(lse_of(s) - mx);
    const float total = mx == -INFINITY ? -INFINITY : mx + logf(sum);
    f32x16 acc[HD / 32];
#pragma unroll
    for (int i = 0; i < HD / 32; ++i) acc[i] = zero16();
    for (int s = 0; s < S; ++s) {
        const float w = total == -INFINITY ? 0.f : expf(lse_of(s) - total);
        const uint64_t *slot = pairs + int64_t(s) * nrow * (HD / 2);
#pragma unroll
        for (int i = 0; i < N; ++i) {
            // (The own slot is read as well, and not used.)
            const f32x2 x = __builtin_bit_cast(
                f32x2, __hip_atomic_load(slot + i * step, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
            f32x16 &t = acc[i / 8];
            t[2 * (i & 7)] = fmaf(w, s == split ? o[i / 8][2 * (i & 7)] : x[0], t[2 * (i & 7)]);
            t[2 * (i & 7) + 1] = fmaf(w, s == split ? o[i / 8][2 * (i & 7) + 1] : x[1], t[2 * (i & 7) + 1]);
        }
    }
#pragma unroll
    for (int i = 0; i < HD / 32; ++i) o[i] = acc[i];
    lse = total;
    return true;
}

template <int HD, bool EXT>
__global__ __launch_bounds__(kKvThreads, 2) void kv_chunk_kernel(const fa_kvcache_args a, const int row_tiles,
                                                                 int32_t *const count, const bool ranked) {
    constexpr int BN = kChunkKeys, TILE = BN * HD * 2, STAGE = 2 * TILE;
    __shared__ __attribute__((aligned(16))) char smem[2 * STAGE];
    __shared__ int pages[kChunkPages];
    __shared__ int ticket;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, hh = lane >> 5;
    const int G = a.nheads / a.nheads_k, R = G * a.seqlen_q, S = a.num_splits;
    TileReader<HD> rd;
    rd.init(lane);
    const int64_t krs = a.k_cache.row_stride, vrs = a.v_cache.row_stride;
    TileCopier<HD, BN, kKvThreads> kcp, vcp;
    kcp.init(krs, wave, lane);
    vcp.init(vrs, wave, lane);
    int rest = blockIdx.x;
    const int rt = rest % row_tiles;
    rest /= row_tiles;
    const int hk = rest % a.nheads_k;
    rest /= a.nheads_k;
    const int split = rest % S;
    const int b = ranked ? a.batch_order[rest / S] : rest / S;

    const KvSeq sq = kv_seq(a, b);
    if (sq.err && a.status && tid == 0) atomicOr(a.status, sq.err);
    const int L = sq.err ? 0 : sq.L0 + a.seqlen_new;
    const int kstart = EXT && a.cache_leftpad ? min(max(a.cache_leftpad[b], 0), L) : 0;

    // This lane's query row (row qpos * G + g of the KV head).
    const int first = rt * kChunkRows, rows_here = min(kChunkRows, R - first);
    const int row = 32 * wave + col;
    const bool row_ok = row < rows_here;
    const int qpos = row_ok ? (first + row) / G : 0;
    const int hq = hk * G + (row_ok ? (first + row) % G : 0);
    const int off = L - a.seqlen_q;  // key position of query 0
    const int qkey = qpos + off;
    // Keys [key_lo, key_hi) a query at key position p sees.  The splits divide
    // the keys that some row of the tile sees, [t_lo, t_hi).
    const int wl = EXT && a.local_window ? a.window_left : -1, wr = EXT && a.local_window ? a.window_right : -1;
    auto key_lo = [&](int p) { return wl >= 0 ? max(kstart, p - wl) : kstart; };
    auto key_hi = [&](int p) {
        int hi = a.causal ? min(L, p + 1) : L;
        if (wr >= 0) hi = min(hi, p + wr + 1);
        return hi;
    };
    const int t_lo = __builtin_amdgcn_readfirstlane(key_lo(first / G + off)), t_n = max(0, key_hi((first + rows_here - 1) / G + off) - t_lo);
    const int s0 = t_lo + int(int64_t(t_n) * split / S), s1 = t_lo + int(int64_t(t_n) * (split + 1) / S);
    const int nb0 = s0 / BN, nb1 = s1 > s0 ? (s1 - 1) / BN + 1 : nb0;
    // Of the split's keys: those the lane's row sees, [lo, hi), those some row
    // of the wave sees and those every row of it sees.
    const int lo = max(s0, key_lo(qkey)), hi = min(s1, key_hi(qkey));
    const int p0w = (first + 32 * wave) / G + off, p1w = (first + min(rows_here, 32 * wave + 32) - 1) / G + off;
    const int any_lo = max(s0, key_lo(p0w)), any_hi = 32 * wave < rows_here ? min(s1, key_hi(p1w)) : s0;
    const int all_lo = max(s0, key_lo(p1w)), all_hi = min(s1, key_hi(p0w));

    const bool neg = a.softmax_scale < 0.f;
    const bool capped = EXT && a.softcap > 0.f, alibi = EXT && a.alibi_slopes != nullptr;
    const bool natural = capped || alibi;  // scores formed in natural units
    const float cscale = natural ? kLog2e : fabsf(a.softmax_scale) * kLog2e;
    const float cap_in = capped ? fabsf(a.softmax_scale) / a.softcap : 0.f;
    const float slope = alibi ? a.alibi_slopes[int64_t(b) * a.alibi_batch_stride + hq] : 0.f;
    const int rpos = sq.L0 + (a.causal || a.local_window ? qpos : 0);  // rotary position
    f16x8 qB[HD / 16];
    {
        const f16 *qp = (const f16 *)a.q.ptr + int64_t(b) * a.q.batch_stride + int64_t(qpos) * a.q.row_stride +
                        int64_t(hq) * a.q.head_stride;
#pragma unroll
        for (int g = 0; g < HD / 16; ++g) {
            u32x4 v = row_ok ? ldg16(qp + 16 * g + 8 * hh) : zero_u4();
            if (EXT && row_ok && 16 * g + 8 * hh < a.rotary_dim) v = rotary8(a, v, qp, 16 * g + 8 * hh, rpos);
            if (neg) v = neg_h8(v);
            qB[g] = as_h8(v);
        }
    }
    // Page ids of the walked keys (this kernel is taken only when they fit).
    const int page = a.page_block_size;
    const int pg0 = a.block_table ? nb0 * BN / page : 0;
    if (a.block_table && nb1 > nb0) {
        const int32_t *bt = a.block_table + int64_t(b) * a.block_table_stride + pg0;
        const int n_pages = (nb1 * BN - 1) / page - pg0 + 1;
        for (int i = tid; i < n_pages; i += kKvThreads) pages[i] = bt[i];
    }
    wait_vmem();  // only the tile copies are in flight in the loop
    __syncthreads();

    const f16 *kc = (const f16 *)a.k_cache.ptr + int64_t(hk) * a.k_cache.head_stride;
    const f16 *vc = (const f16 *)a.v_cache.ptr + int64_t(hk) * a.v_cache.head_stride;
    auto issue = [&](int nb) FA_INLINE {
        int64_t blk = sq.row;
        int at = nb * BN;  // token within the cache row or page
        if (a.block_table) {
            const int pi = at / page;
            blk = __builtin_amdgcn_readfirstlane(pages[pi - pg0]);
            at -= pi * page;
        }
        const f16 *kb = kc + blk * a.k_cache.batch_stride + int64_t(at) * krs;
        const f16 *vb = vc + blk * a.v_cache.batch_stride + int64_t(at) * vrs;
        const int soff = (nb & 1) * STAGE;
        if ((!EXT || nb * BN >= t_lo) && nb * BN + BN <= L) {
            kcp.template copy_to<true>(lds_addr(smem) + soff, kb, krs);
            vcp.template copy_to<true>(lds_addr(smem) + soff + TILE, vb, vrs);
        } else {  // keys past L re-read key L - 1, keys that no row sees at the start re-read the first seen one (masked)
            dma_tile<HD, BN, kKvThreads>(smem + soff, kb, krs, 0, L - 1 - nb * BN, wave, lane, t_lo - nb * BN);
            dma_tile<HD, BN, kKvThreads>(smem + soff + TILE, vb, vrs, 0, L - 1 - nb * BN, wave, lane, t_lo - nb * BN);
        }
    };

    f32x16 o[HD / 32];
#pragma unroll
    for (int i = 0; i < HD / 32; ++i) o[i] = zero16();
    float m_t = -INFINITY, l_p = 0.f;
    if (nb1 > nb0) issue(nb0);
    for (int nb = nb0; nb < nb1; ++nb) {
        wait_vmem();
        __syncthreads();  // block nb is in LDS; every wave is done with the other stage
        if (nb + 1 < nb1) issue(nb + 1);
        const int p0 = nb * BN;
        if (p0 >= any_hi || p0 + BN <= any_lo) continue;  // no key for this wave
        // The lane's read bases with this block's stage added (opaque, so the
        // per-read addresses are not hoisted to hold registers; see TileReader).
        const int soff = (nb & 1) * STAGE;
        int ab = rd.a_base + soff, tb0 = rd.tr_base[0] + soff, tb1 = rd.tr_base[1] + soff;
        asm volatile("" : "+v"(ab), "+v"(tb0), "+v"(tb1));
        f32x16 s[2];
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
            s[kt] = zero16();
#pragma unroll
            for (int g = 0; g < HD / 16; ++g)
                s[kt] = mfma32(rd.a_operand_at(smem + 32 * kt * (HD * 2), ab, g), qB[g], s[kt]);
        }
        if constexpr (EXT) {
            if (natural) {
                const float sc = fabsf(a.softmax_scale);
                const float dist0 = float(qkey - p0 - 8 * hh);
#pragma unroll
                for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        float x = capped ? a.softcap * tanh_fast(s[kt][r] * cap_in) : s[kt][r] * sc;
                        if (alibi) x -= slope * fabsf(dist0 - float(kt * 32 + acc_lrow(r, 0)));
                        s[kt][r] = x;
                    }
            }
        }
        if (p0 < all_lo || p0 + BN > all_hi) {
            const int lo_c = lo - p0 - 8 * hh, hi_c = hi - p0 - 8 * hh;
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int c = kt * 32 + acc_lrow(r, 0);
                    if (c < lo_c || c >= hi_c) s[kt][r] = -INFINITY;
                }
        }
        float mx = s[0][0];
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[kt][r]);
        mx = max_xor32(mx);
        const float mx_t = mx == -INFINITY ? -INFINITY : mx * cscale;
        if (__builtin_amdgcn_ballot_w64(mx_t > m_t + kKvRescaleSlack) != 0) {
            const float m_new = fmaxf(m_t, mx_t);
            const float alpha = m_new == -INFINITY ? 1.f : exp2_fast(m_t - m_new);
            l_p *= alpha;
#pragma unroll
            for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
            m_t = m_new;
        }
        const float m_use = m_t == -INFINITY ? 0.f : m_t;
        float rs = 0.f;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float p = exp2_fast(fmaf(s[kt][r], cscale, -m_use));
                s[kt][r] = p;
                rs += p;
            }
        l_p += rs;
        float minus1 = -1.f;
        asm("" : "+v"(minus1));
#pragma unroll
        for (int gg = 0; gg < 4; ++gg) {
            f16x8 pl;
            u32x4 hi4 = __builtin_bit_cast(u32x4, pack8(s[gg >> 1], 8 * (gg & 1)));
            asm("" : "+v"(hi4));  // opaque: the halves below come from the packed words, not from conversions of their own
            const f16x8 ph = as_h8(hi4);
#pragma unroll
            for (int u = 0; u < 8; ++u) pl[u] = (f16)fmaf(float(ph[u]), minus1, s[gg >> 1][8 * (gg & 1) + u]);
#pragma unroll
            for (int dt = 0; dt < HD / 32; ++dt) {
                const f16x8 va = rd.tr_operand_at(smem + TILE + 16 * gg * (HD * 2), tb0, tb1, dt);
                o[dt] = mfma32(va, ph, o[dt]);
                o[dt] = mfma32(va, pl, o[dt]);
            }
        }
    }

    const float l_tot = sum_xor32(l_p);
    const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    float lse = l_tot > 0.f ? (m_t + log2_fast(l_tot)) * kLn2 : -INFINITY;
#pragma unroll
    for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] *= inv;
    const int64_t tile = (int64_t(b) * a.nheads_k + hk) * row_tiles + rt;
    const int64_t row0 = (int64_t(b) * a.nheads_k + hk) * R + first;
    // Opaque to the optimiser: the row's output addresses are formed here, not
    // before the block loop and held through it.
    int orow = row;
    asm volatile("" : "+v"(orow));
    if (S == 1 || chunk_merge<HD>(a, count + tile, split, row0, rows_here, orow, hh, &ticket, o, lse)) {
        if (orow < rows_here) {
            const int oq = (first + orow) / G, oh = hk * G + (first + orow) % G;
            f16 *op = (f16 *)a.o.ptr + int64_t(b) * a.o.batch_stride + int64_t(oq) * a.o.row_stride +
                      int64_t(oh) * a.o.head_stride;
#pragma unroll
            for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
                for (int a4 = 0; a4 < 4; ++a4) {
                    f16x4 v;
#pragma unroll
                    for (int t = 0; t < 4; ++t) v[t] = (f16)o[dt][4 * a4 + t];
                    *reinterpret_cast<f16x4 *>(op + dt * 32 + 8 * a4 + 4 * hh) = v;
                }
            if (hh == 0)
                a.lse[(int64_t(b) * a.nheads + oh) * a.seqlen_q + oq] = lse == -INFINITY ? 0.f : lse;
        }
    }
}

// ---------------------------------------------------------------------------
// Combine kernel: one wave per (batch, head, qpos) row.
template <int HD>
__global__ __launch_bounds__(256) void kv_combine_kernel(const fa_kvcache_args a) {
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= a.batch * a.nheads * a.seqlen_q) return;
    combine_rows<HD, false, 1, kPreSplits>(a, {r}, 1, threadIdx.x & 63);
}

static int check_kv(const fa_kvcache_args *p) {
    if (!p) return FA_ERR_INVALID_ARG;
    const fa_kvcache_args &a = *p;
    if (a.head_dim != 64 && a.head_dim != 128) return FA_ERR_UNSUPPORTED;
    if (a.batch < 0 || a.seqlen_q < 0 || a.nheads <= 0 || a.nheads_k <= 0 || a.nheads % a.nheads_k != 0 ||
        a.seqlen_new < 0 || a.num_splits < 1 || !a.cache_seqlens || !a.lse)
        return FA_ERR_INVALID_ARG;
    if (a.block_table && (a.page_block_size <= 0 || a.page_block_size % kTile != 0)) return FA_ERR_INVALID_ARG;
    if (a.block_table && a.cache_batch_idx) return FA_ERR_INVALID_ARG;
    if (!(a.softcap >= 0.f) || a.softcap == INFINITY) return FA_ERR_INVALID_ARG;  // NaN fails too
    if (a.rotary_dim != 0 &&
        (a.rotary_dim < 0 || a.rotary_dim % 16 != 0 || a.rotary_dim > a.head_dim || a.rotary_seqlen < 1 ||
         !a.rotary_cos || !a.rotary_sin || !a.k_new.ptr ||
         ((reinterpret_cast<uintptr_t>(a.rotary_cos) | reinterpret_cast<uintptr_t>(a.rotary_sin)) & 15u)))
        return FA_ERR_INVALID_ARG;
    return FA_OK;
}

// Whether many query rows (tiles of 128 rows over all sequences and KV heads) are
// kv_chunk_kernel's: there are enough tiles that few splits fill the chip, few keys
// to split, or so many that merging more splits does not weigh.  Otherwise (one or
// two KV heads, few sequences) kv_splitkv_kernel's four waves share a tile's keys
// and its many items merge faster.  natural: scores formed in natural units (softcap,
// ALiBi), whose arithmetic costs this kernel more than the shared loads save.
// Measured on MI355X, us a call at each kernel's own splits, split kernel -> this one
// (tiles):
//   64/1 heads, 1 token, 5.5k keys (1): 39 -> 53       128/1, 1 x 210k (1): 181 -> 351
//   32/2, 8 tokens, 7.8k (2): 38 -> 48                 b4 8/1, 16 x 63k (4): 60 -> 101
//   32/8, 16 x 18k (8): 52 -> 60                       64/4, 9 x 20k (8): 67 -> 71
//   32/8, 32 x 106k (8): 274 -> 165                    64/2, 9 x 186k (6): 318 -> 211
//   12 - 16 tiles: 1.0 - 1.9x faster; 17 and more: 1.2 - 1.9x; up to 4k keys: 1.0 - 1.4x
//   natural: b4 16/1, 8 x 15k (4): 54 -> 86; 16 tiles: 0.77 - 1.3x; 1 - 8 tiles on 2k - 4k
//   keys: 0.84 - 0.9x; on up to 1k: 1.07 - 1.26x
static bool chunk_pays(int64_t tiles, int64_t keys, bool natural, int num_cus) {
    const int64_t cus = std::max(num_cus, 1);
    if (natural) return 16 * tiles > cus || (keys > 0 && keys <= 1024);
    return 24 * tiles > cus || (keys > 0 && keys <= 4096) || (48 * tiles > cus && keys >= 65536);
}

// Splits of the many-row kernel: the fewest key blocks on the busiest CU (a CU
// with one workgroup is about 10 % slower per block) and 1.3 blocks' time for
// every split to merge.  Measured on MI355X with 32 / 8 heads, head_dim 128, us
// per call at 1 split -> the splits taken: 512 rows x 1 sequence of 8k keys
// 226 -> 128 (4 splits), 128 x 1 x 8k 214 -> 59 (8), 32 x 8 x 8k 215 -> 82 (4),
// 1024 x 1 x 15k 444 -> 410 (2).  At most 16 where there are enough tiles for those
// to fill the chip (chunk_pays), 32 otherwise.
static int chunk_num_splits(int64_t tiles, int64_t keys, int num_cus) {
    const int64_t cus = std::max(num_cus, 1);
    const double blocks = (double(keys) + kChunkKeys - 1) / kChunkKeys;
    const int most = 24 * tiles > cus ? 16 : kChunkMaxSplits;
    int best = 1;
    double best_t = 0;
    for (int S = 1; S <= most && (S == 1 || blocks >= 4 * S); ++S) {
        const int64_t wgs = tiles * S;
        double t = double((wgs + cus - 1) / cus) * blocks / S;
        if (wgs <= cus) t *= 1.1;
        t += 1.3 * (S - 1);
        if (S == 1 || t < best_t) {
            best = S;
            best_t = t;
        }
    }
    return best;
}

static int64_t chunk_tiles(const fa_kvcache_args &a) {
    return int64_t(a.batch) * a.nheads_k * (((a.nheads / a.nheads_k) * a.seqlen_q + kChunkRows - 1) / kChunkRows);
}
static int64_t chunk_items(const fa_kvcache_args &a) { return chunk_tiles(a) * a.num_splits; }

// Key positions a call's splits divide at most (the live lengths are on the
// device): with a left window, the window and the call's own tokens (64 sequences
// of 1k - 16k tokens, 4096-key window: 192 us in the 2 splits of the whole capacity,
// 182 in 1).
static int64_t split_keys(const fa_kvcache_args &a) {
    const int64_t keys = a.cache_capacity;
    return a.local_window && a.window_left >= 0 ? std::min<int64_t>(keys, int64_t(a.window_left) + 1 + a.seqlen_q) : keys;
}

// Scratch bytes fa_fwd_kvcache_noalloc needs for a call: the split accumulators, then
// batch + 1 int32s of order and counter, then the split counts.
static size_t noalloc_bytes(const fa_kvcache_args &a) {
    return fa_kv_workspace_bytes(&a) +
           (size_t(a.batch > 0 ? a.batch : 0) + 1 + size_t(fa_kv_split_count_len(&a))) * sizeof(int32_t);
}

// Whether kv_chunk_kernel suits a call, if it is given the workspaces that the
// kernel needs: at least 64 query rows per KV head (with 64 rows, 8 sequences of 8k
// keys, 32 / 8 heads: 71 us against 114 at the best split counts; with 32 rows the
// other kernel reads K and V once as well and its waves share the keys) in enough
// tiles (chunk_pays).  Its 64-key blocks must not straddle pages, and its page ids fit
// in LDS.
static bool chunk_suits(const fa_kvcache_args &a, int num_cus) {
    if ((a.nheads / a.nheads_k) * a.seqlen_q < kChunkMinRows) return false;
    if (a.block_table && (a.page_block_size % kChunkKeys != 0 || a.cache_capacity <= 0 ||
                          a.cache_capacity / a.page_block_size > kChunkPages))
        return false;
    return chunk_pays(chunk_tiles(a), split_keys(a), a.softcap > 0.f || a.alibi_slopes, num_cus);
}

}  // namespace fa

extern "C" int fa_kv_args_num_splits(const fa_kvcache_args *args, int requested, int num_cus) {
    // An explicit request is honoured (kvcache_native.cu:922-924).  Otherwise
    // (measured on MI355X over paged and contiguous decode shapes) a work item
    // streams best with about 8192 cache positions: fewer and the per-item
    // start-up and the combine weigh in, more and the longest-first deal
    // balances worse.  Enough splits are also taken for one item per compute
    // unit, and a split keeps at least 512 positions, or, for a cache of 512
    // positions or more cut into at most 16 splits, at least 64 (a short cache
    // on few sequences: one sequence of 1024 positions, 32 / 8 heads, takes
    // 15.5 us per call in 16 splits against 20.3 in 2).  Only the capacity is
    // known on the host (the live lengths are on the device).
    if (requested > 0) return requested;
    if (!args || args->batch <= 0 || args->nheads_k <= 0 || args->nheads <= 0) return 1;
    const fa_kvcache_args &a = *args;
    const int64_t keys = fa::split_keys(a);
    if (keys <= 0) return 1;
    if (fa::chunk_suits(a, num_cus)) return fa::chunk_num_splits(fa::chunk_tiles(a), keys, num_cus);
    const int rows = (a.nheads / a.nheads_k) * a.seqlen_q;
    const int64_t wgs = int64_t(a.batch) * a.nheads_k * ((rows + 31) / 32);
    const int64_t by_len = (keys + 4096) / 8192;
    const int64_t by_fill = (int64_t(std::max(num_cus, 1)) + wgs - 1) / std::max<int64_t>(wgs, 1);
    int64_t max_by_len = keys / 512;
    if (keys >= 512) max_by_len = std::max<int64_t>(max_by_len, std::min<int64_t>(16, keys / 64));
    max_by_len = std::max<int64_t>(1, max_by_len);
    // One workgroup combines the splits of a tile's 32 rows: with many rows on few
    // tiles that outweighs idle CUs (us in the splits that fill the chip -> 16: 64/1
    // heads, 1 token on 70k keys 128: 271 -> 80; b2 16/1 d64, 4 tokens on 39k keys 64:
    // 120 -> 45; at 225k keys b3 128/1 d64 254 in 16, 187 in 32).
    const int64_t most = rows < fa::kChunkMinRows ? 128 : keys > 131072 ? 32 : 16;
    return int(std::max<int64_t>(1, std::min<int64_t>({std::max(by_len, by_fill), max_by_len, most})));
}

extern "C" int fa_kv_num_splits(int requested, int seqlen_k_capacity, int head_dim, int seqlen_q, int batch,
                                int nheads, int nheads_k, int num_cus) {
    // The same for a call without options on a cache whose pages are multiples of
    // 64 tokens, in no more splits than the static scratch of
    // fa_fwd_kvcache_noalloc holds where many rows ask for more (a count from here
    // always suits that entry there).
    fa_kvcache_args a{};
    a.cache_capacity = seqlen_k_capacity;
    a.head_dim = head_dim;
    a.seqlen_q = seqlen_q;
    a.batch = batch;
    a.nheads = nheads;
    a.nheads_k = nheads_k;
    a.num_splits = fa_kv_args_num_splits(&a, requested, num_cus);
    if (requested <= 0 && a.num_splits > 1 && fa::chunk_suits(a, num_cus))
        while (a.num_splits > 1 && fa::noalloc_bytes(a) > FA_NOALLOC_SCRATCH_BYTES) --a.num_splits;
    return a.num_splits;
}

extern "C" size_t fa_kv_workspace_bytes(const fa_kvcache_args *a) {
    if (!a || a->num_splits <= 1) return 0;
    const size_t rows = size_t(a->batch) * a->nheads * a->seqlen_q;
    return size_t(a->num_splits) * rows * (size_t(a->head_dim) + 1) * sizeof(float);
}

extern "C" size_t fa_kv_split_count_len(const fa_kvcache_args *a) {
    if (!a || a->num_splits <= 1 || a->batch <= 0 || a->nheads_k <= 0 || a->nheads <= 0 || a->seqlen_q <= 0)
        return 0;
    const int64_t rows = int64_t(a->nheads / a->nheads_k) * a->seqlen_q;
    return size_t(int64_t(a->batch) * a->nheads_k * ((rows + 31) / 32));
}

namespace fa {
namespace {

bool has_append(const fa_kvcache_args &a) { return a.k_new.ptr && a.seqlen_new > 0 && a.batch > 0; }

int check_append(const fa_kvcache_args &a) {
    if (!has_append(a)) return FA_OK;
    if (!a.v_new.ptr || fa::check_tensor(a.k_new, true) || fa::check_tensor(a.v_new, true) ||
        fa::check_tensor(a.k_cache, true) || fa::check_tensor(a.v_cache, true))
        return FA_ERR_INVALID_ARG;
    return FA_OK;
}

// Work items of the split kernel: (batch, kv head, split, 32-row tile).
int64_t split_items(const fa_kvcache_args &a) {
    const int R = (a.nheads / a.nheads_k) * a.seqlen_q;
    return int64_t(a.batch) * a.nheads_k * ((R + 31) / 32) * a.num_splits;
}

int check_split(const fa_kvcache_args &a) {
    if (fa::check_tensor(a.q, true) || fa::check_tensor(a.o, true) || fa::check_tensor(a.k_cache, true) ||
        fa::check_tensor(a.v_cache, true))
        return FA_ERR_INVALID_ARG;
    if (a.num_splits > 1 && (!a.out_accum || !a.lse_accum)) return FA_ERR_WORKSPACE;
    // The combine reads head_dim 128 partials as 64-bit (atomic) loads.
    if (a.num_splits > 1 && (reinterpret_cast<uintptr_t>(a.out_accum) & 7u)) return FA_ERR_INVALID_ARG;
    if (split_items(a) > 0x7fffffff) return FA_ERR_INVALID_ARG;
    return FA_OK;
}

// The split kernel combines its partials itself: a resident grid (batch_order)
// with split counts and more than one split.
bool fused_combine(const fa_kvcache_args &a) { return a.batch_order && a.split_count && a.num_splits > 1; }

// KV heads per work item of the resident split kernel without options: in a
// head-interleaved cache (head stride = head_dim) enough adjacent heads that
// one key position's rows of an item are 512 contiguous bytes (HBM reads of
// 128-byte pieces at a 2 KB stride run about 10 % below 512-byte ones on
// MI355X), while every resident workgroup still gets at least four items:
// with fewer, the items of the longest sequences (their splits are the
// largest) decide the call's time.
int kv_heads_per_item(const fa_kvcache_args &a) {
    const bool interleaved = a.k_cache.head_stride == a.head_dim && a.v_cache.head_stride == a.head_dim;
    const bool ext = a.local_window || a.softcap > 0.f || a.cache_leftpad || a.alibi_slopes || a.rotary_dim > 0;
    if (!a.batch_order || ext || !interleaved) return 1;
    const int64_t items = split_items(a), slots = 2 * int64_t(device_cus());
    int hpi = 1;
    while (hpi < 4 && int64_t(a.head_dim) * 2 * (2 * hpi) <= 512 && a.nheads_k % (2 * hpi) == 0 &&
           items / (2 * hpi) >= 4 * slots)
        hpi *= 2;
    return hpi;
}

// Whether the split kernel of a call is kv_chunk_kernel: it suits the call, there
// are few enough splits for one workgroup to merge, and the split counts to do it
// with.
bool use_chunk(const fa_kvcache_args &a) {
    return a.batch_order && a.num_splits <= kChunkMaxSplits && (a.num_splits == 1 || a.split_count) &&
           chunk_suits(a, device_cus());
}

// Whether the split kernel's items come in the order of batch_order: there are
// more of them than CUs.
bool kv_ranked(const fa_kvcache_args &a) {
    const int64_t n = use_chunk(a) ? chunk_items(a) : split_items(a) / kv_heads_per_item(a);
    return a.batch_order && n > int64_t(device_cus());
}

// kv_prep_kernel over the append's chunks (append) after one ordering workgroup (order).
int launch_prep(const fa_kvcache_args &a, bool append, bool order, hipStream_t s) {
    const int64_t chunks = append ? int64_t(a.batch) * a.seqlen_new * a.nheads_k * (a.head_dim / 8) : 0;
    int32_t *count = order && fused_combine(a) ? a.split_count : nullptr;
    const int n_count = count ? int(fa_kv_split_count_len(&a)) : 0;
    const bool rank = order && kv_ranked(a);
    const int order_wgs = rank || count ? 1 : 0;
    const int64_t blocks = order_wgs + (chunks + kOrderThreads - 1) / kOrderThreads;
    if (blocks == 0) return FA_OK;
    if (blocks > 0x7fffffff) return FA_ERR_INVALID_ARG;
    if (a.head_dim == 128)
        hipLaunchKernelGGL(kv_prep_kernel<128>, dim3(unsigned(blocks)), dim3(kOrderThreads), 0, s, a, order_wgs, rank, count,
                           n_count);
    else
        hipLaunchKernelGGL(kv_prep_kernel<64>, dim3(unsigned(blocks)), dim3(kOrderThreads), 0, s, a, order_wgs, rank, count,
                           n_count);
    return int(hipGetLastError());
}

int launch_chunk(const fa_kvcache_args &a, hipStream_t s) {
    const int row_tiles = ((a.nheads / a.nheads_k) * a.seqlen_q + kChunkRows - 1) / kChunkRows;
    const int64_t n = chunk_items(a);
    if (n == 0) return FA_OK;
    const bool ranked = kv_ranked(a), ext = a.local_window || a.softcap > 0.f || a.cache_leftpad || a.alibi_slopes || a.rotary_dim > 0;
    auto go = [&](auto hd_tag, auto ext_tag) {
        hipLaunchKernelGGL((kv_chunk_kernel<decltype(hd_tag)::value, decltype(ext_tag)::value>), dim3(unsigned(n)),
                           dim3(kKvThreads), 0, s, a, row_tiles, a.split_count, ranked);
    };
    using H128 = std::integral_constant<int, 128>;
    using H64 = std::integral_constant<int, 64>;
    if (a.head_dim == 128)
        ext ? go(H128{}, std::true_type{}) : go(H128{}, std::false_type{});
    else
        ext ? go(H64{}, std::true_type{}) : go(H64{}, std::false_type{});
    return int(hipGetLastError());
}

// The split kernel.  With batch_order: a resident grid of two workgroups per CU
// that deals the items out, in its order where launch_prep on the same stream has
// ranked the sequences and reset the counter (kv_ranked: more items than CUs; else
// each workgroup has one item).  Without it: one workgroup per item.
int launch_split(const fa_kvcache_args &a, hipStream_t s) {
    if (use_chunk(a)) return launch_chunk(a, s);
    const int hpi = kv_heads_per_item(a);
    const int64_t gx = split_items(a) / hpi;
    if (gx == 0) return FA_OK;
    const int row_tiles = ((a.nheads / a.nheads_k) * a.seqlen_q + 31) / 32;
    const int n_items = int(gx);
    const bool dyn = a.batch_order != nullptr;
    const unsigned grid = unsigned(dyn ? std::min<int64_t>(gx, 2 * int64_t(device_cus())) : gx);
    int32_t *count = fused_combine(a) ? a.split_count : nullptr;
    const bool ranked = kv_ranked(a);
    const bool ext = a.local_window || a.softcap > 0.f || a.cache_leftpad || a.alibi_slopes || a.rotary_dim > 0;
    auto go = [&](auto hd_tag, auto dyn_tag, auto ext_tag, auto hpi_tag) {
        constexpr int HD = decltype(hd_tag)::value, HPI = decltype(hpi_tag)::value;
        constexpr bool DYN = decltype(dyn_tag)::value, EXT = decltype(ext_tag)::value;
        hipLaunchKernelGGL((kv_splitkv_kernel<HD, DYN, EXT, HPI>), dim3(grid), dim3(kKvThreads), 0, s, a, row_tiles,
                           n_items, count, ranked);
    };
    using H128 = std::integral_constant<int, 128>;
    using H64 = std::integral_constant<int, 64>;
    using P1 = std::integral_constant<int, 1>;
    using P2 = std::integral_constant<int, 2>;
    using P4 = std::integral_constant<int, 4>;
    using T = std::true_type;
    using F = std::false_type;
    if (a.head_dim == 128) {
        if (dyn && !ext) hpi == 2 ? go(H128{}, T{}, F{}, P2{}) : go(H128{}, T{}, F{}, P1{});
        else if (dyn) go(H128{}, T{}, T{}, P1{});
        else ext ? go(H128{}, F{}, T{}, P1{}) : go(H128{}, F{}, F{}, P1{});
    } else {
        if (dyn && !ext) hpi == 4 ? go(H64{}, T{}, F{}, P4{}) : hpi == 2 ? go(H64{}, T{}, F{}, P2{}) : go(H64{}, T{}, F{}, P1{});
        else if (dyn) go(H64{}, T{}, T{}, P1{});
        else ext ? go(H64{}, F{}, T{}, P1{}) : go(H64{}, F{}, F{}, P1{});
    }
    return int(hipGetLastError());
}

// The combine kernel, unless there is one split or the split kernel combined.
int launch_combine(const fa_kvcache_args &a, hipStream_t s) {
    if (a.num_splits <= 1 || fused_combine(a)) return FA_OK;
    const int64_t nrow = int64_t(a.batch) * a.nheads * a.seqlen_q;
    if (nrow == 0) return FA_OK;
    const int64_t blocks = (nrow + 3) / 4;
    if (a.head_dim == 128)
        hipLaunchKernelGGL(kv_combine_kernel<128>, dim3(unsigned(blocks)), dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL(kv_combine_kernel<64>, dim3(unsigned(blocks)), dim3(256), 0, s, a);
    return int(hipGetLastError());
}

}  // namespace
}  // namespace fa

extern "C" int fa_kv_append(const fa_kvcache_args *args, void *stream) {
    int rc = fa::check_kv(args);
    if (rc || (rc = fa::check_append(*args))) return rc;
    if (!fa::has_append(*args)) return FA_OK;
    return fa::launch_prep(*args, true, false, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int fa_kv_splitkv(const fa_kvcache_args *args, void *stream) {
    int rc = fa::check_kv(args);
    if (rc || (rc = fa::check_split(*args))) return rc;
    const fa_kvcache_args &a = *args;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (fa::split_items(a) == 0) return FA_OK;
    if (a.batch_order && (rc = fa::launch_prep(a, false, true, s))) return rc;
    return fa::launch_split(a, s);
}

extern "C" int fa_kv_combine(const fa_kvcache_args *args, void *stream) {
    int rc = fa::check_kv(args);
    if (rc) return rc;
    const fa_kvcache_args &a = *args;
    if (a.num_splits <= 1 || fa::fused_combine(a)) return FA_OK;
    if (!a.out_accum || !a.lse_accum) return FA_ERR_WORKSPACE;
    return fa::launch_combine(a, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int fa_fwd_kvcache(const fa_kvcache_args *args, void *stream) {
    int rc = fa::check_kv(args);
    if (rc || (rc = fa::check_append(*args)) || (rc = fa::check_split(*args))) return rc;
    const fa_kvcache_args &a = *args;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    // One launch appends and ranks (the ranking reads cache_seqlens only).
    const bool order = a.batch_order && fa::split_items(a) > 0;
    if ((rc = fa::launch_prep(a, fa::has_append(a), order, s))) return rc;
    if ((rc = fa::launch_split(a, s))) return rc;
    return fa::launch_combine(a, s);
}

// ---------------------------------------------------------------------------
// Allocation-free decode: fa_fwd_kvcache with its split workspace (out_accum,
// lse_accum, batch_order, split_count) carved from a static device array
// instead of caller memory, for callers that cannot allocate (code under HIP
// graph capture, serving loops, harnesses that forbid hipMalloc).  The array
// is FA_NOALLOC_SCRATCH_BYTES per device for the life of the process; its
// device address is looked up once per device (hipGetSymbolAddress) and only
// that address is handed to the kernels.  Nothing in it needs clearing between
// calls: the split kernel writes every partial it later combines, and the
// ordering workgroup resets the work counter and the split counts.  Calls on
// one device share the array, so calls that overlap on a device (different
// streams) race; their results are undefined, but no workgroup waits for another
// one's counts, so every kernel ends.
static __device__ __align__(256) char scratch[FA_NOALLOC_SCRATCH_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch[kMaxDevices] = {};

// Device address of this device's scratch array (looked up on the device's first call).
int scratch_address(void **out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return int(e);
    if (dev < 0 || dev >= kMaxDevices) return FA_ERR_INVALID_ARG;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[dev]) {
        // The first call on a device may come from inside a stream capture whose
        // mode forbids runtime calls that are not stream work (the lookup can
        // load the code object on the device): relax this thread's mode for the
        // lookup only; it enqueues nothing.
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        e = hipThreadExchangeStreamCaptureMode(&mode);
        if (e != hipSuccess) return int(e);
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        const hipError_t e2 = hipThreadExchangeStreamCaptureMode(&mode);
        if (e != hipSuccess) return int(e);
        if (e2 != hipSuccess) return int(e2);
        if (!p) return FA_ERR_SCRATCH;
        g_scratch[dev] = p;
    }
    *out = g_scratch[dev];
    return FA_OK;
}

}  // namespace

extern "C" int fa_fwd_kvcache_noalloc(const fa_kvcache_args *args, void *stream) {
    int rc = fa::check_kv(args);
    if (rc) return rc;
    if (fa::noalloc_bytes(*args) > FA_NOALLOC_SCRATCH_BYTES) return FA_ERR_SCRATCH;
    void *base = nullptr;
    if ((rc = scratch_address(&base))) return rc;
    fa_kvcache_args a = *args;
    const size_t acc = fa_kv_workspace_bytes(&a);
    float *f = static_cast<float *>(base);
    if (a.num_splits > 1) {
        a.out_accum = f;
        a.lse_accum = f + size_t(a.num_splits) * a.batch * a.nheads * a.seqlen_q * a.head_dim;
    } else {
        a.out_accum = a.lse_accum = nullptr;
    }
    a.batch_order = reinterpret_cast<int32_t *>(static_cast<char *>(base) + acc);
    a.split_count = fa_kv_split_count_len(&a) > 0 ? a.batch_order + (a.batch > 0 ? a.batch : 0) + 1 : nullptr;
    return fa_fwd_kvcache(&a, stream);
}
