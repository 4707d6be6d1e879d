// Forward attention for gfx950 (MI355X).
//
// Replaces the reference forward (csrc/flash_attn/src/flash_fwd_kernel.h:23-711,
// flash_fwd_launch_template.h:9-118).  Semantics kept: fp16 Q/K/V, fp32
// accumulation, scale applied to the fp32 scores, bottom-right causal mask
// (mask.h:52-104), GQA head mapping (fwd_kernel.h:76), varlen offsets and
// seqused_k (block_info.h:4-36), P rounded to fp16 before the PV product
// (fwd_kernel.h:415), O = 0 and LSE = 0 for a row with no visible key
// (fwd_kernel.h:616-662).
//
// Each wave owns 32 queries of one (batch, head) and walks 64-key blocks.  It
// computes S^T = K Q^T (keys on the MFMA M dimension) so each lane holds one
// query column and 32 keys of a block: the row max needs one cross-half
// exchange and the row sum none.  Q^T stays in registers as the B operand.  K
// and V tiles go from HBM straight into LDS with global_load_lds (no register
// staging), two stages; V keeps its natural layout and is read transposed
// with ds_read_b64_tr_b16.  P^T feeds the O^T += V^T P^T MFMAs directly from
// the accumulators (see fa_common.h).
//
// Two kernels share that per-wave arithmetic and differ in how the waves of a
// SIMD take turns.  With one wave group, which walks a row's key blocks in order,
// their results are the same bit for bit; two groups and splits round and sum in
// another order, so on small grids a row's bits depend on the plan, that is on
// batch, head count and lengths (fwd_plan), but not on how GQA heads are packed:
//   * fwd_pp_kernel (head_dim 128, grids of at least two workgroups per CU):
//     8 waves, two per SIMD, in two groups that alternate a matrix phase (the
//     PV product of block j - 1 and the S product of block j: all the LDS
//     operand reads and MFMAs) and a softmax phase (block j's exponentials),
//     separated by workgroup barriers, so one group's softmax runs on the
//     VALU while the other group's MFMAs run on the matrix cores;
//   * fwd_kernel (head_dim 64 and small grids): 4 waves, two (head_dim 128)
//     or three (head_dim 64) independent workgroups per CU; on grids too small
//     for that, two groups of 4 or 2 waves per workgroup, and several workgroups
//     per query block, share the key blocks (fwd_plan).
#include <type_traits>

#include "fa_common.h"

namespace fa {

constexpr int kFwdBN = 64;  // keys per block

template <int HD, int NT>
struct FwdCfg {
    static constexpr int BM = 32 * (NT / 64);     // queries per workgroup (32 per wave)
    static constexpr int BN = kFwdBN;
    static constexpr int TILE = BN * HD * 2;      // one K or V tile
    static constexpr int STAGE = 2 * TILE;        // a K tile and a V tile
};

// Each row's probabilities P = exp2(S*c - m) are taken against its exact
// running maximum m, as in the reference's online softmax: the block that
// raises some row's maximum rescales O and the row sums of the wave (by 1 for
// the rows whose maximum stands), so a row's largest score gives P = 1 exactly
// and no P exceeds 1.  (Raising m only when a score outgrows it by 2^8 skips
// most rescales but rounds the dominant keys' P to fp16 at up to 2^8, which
// doubles the output error of rows dominated by a few keys.)  As in the
// reference, the PV product takes P rounded to fp16 and both O and the LSE
// are normalised by the fp32 sum of the unrounded P.

// Per-workgroup extents and base pointers of one (batch, query heads, block of
// query positions).  A workgroup covers gp = 2^lg query heads of one GQA group
// (gp divides the group, so the heads share their K / V) at P = BM / gp
// positions from m0: its K / V tiles serve all of them.  Each wave takes 32
// rows of one head (fwd_wave narrows the pointers to it).
struct FwdWork {
    int b, h, hk, sq, sk, m0, P, causal_off, n_blocks;
    const f16 *qp, *kp, *vp;
    f16 *op;
    float *lse_row;
    float cscale;
    bool neg;
};

// Fills w for workgroup bid (of the unsplit grid); false when the block has no query rows
// (its LSE padding is then written here).
template <int BM, bool CAUSAL>
__device__ __forceinline__ bool fwd_work(const fa_fwd_args &a, int num_m_blocks, int lg, int bid, FwdWork &w) {
    int mb;
    const int gp = 1 << lg;
    const int packs = a.nheads >> lg;  // head packs per batch
    if (a.work_order && a.cu_seqlens_q) {
        // Item of the device-built order (head packs fastest), longest first.
        const int it = a.work_order[bid / packs];
        w.b = __builtin_amdgcn_readfirstlane(it / num_m_blocks);
        mb = __builtin_amdgcn_readfirstlane(it - w.b * num_m_blocks);
        w.h = (bid % packs) * gp;
    } else {
        const int bp_count = a.batch * packs;
        const int bp = bid % bp_count;
        mb = bid / bp_count;
        if (CAUSAL) mb = num_m_blocks - 1 - mb;  // causal blocks are issued heaviest first
        w.b = bp / packs;
        w.h = (bp - w.b * packs) * gp;
    }
    w.P = BM >> lg;
    w.hk = w.h / (a.nheads / a.nheads_k);
    const bool packed_q = a.cu_seqlens_q != nullptr, packed_k = a.cu_seqlens_k != nullptr;
    const SeqInfo si = seq_info(w.b, a.seqlen_q, a.seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k, a.seqused_k,
                                a.seqused_k_add);
    w.sq = si.sq;
    w.sk = si.sk;
    int kb = a.k_batch_idx ? a.k_batch_idx[w.b] : w.b;
    if (a.seqused_k) {
        // KV-cache chunk: a key count past the cache or a cache row outside it
        // leaves the batch with no keys, and the error goes to the status word.
        const int used = a.seqused_k[w.b];
        const int err = (used < 0 || int64_t(used) + a.seqused_k_add > a.seqlen_k ? 1 : 0) |
                        (a.k_batch_idx && a.k_batch > 0 && (kb < 0 || kb >= a.k_batch) ? 2 : 0);
        if (err) {
            w.sk = 0;
            kb = 0;
            if (a.status && threadIdx.x == 0) atomicOr(a.status, err);
        }
    }
    w.m0 = mb * w.P;
    w.lse_row = a.lse + (int64_t(w.b) * a.nheads + w.h) * a.lse_seqlen;
    if (w.m0 >= w.sq) {
        // Rows past this sequence's length: LSE padding is 0 (flash_api.cpp:388).
        for (int i = threadIdx.x; i < gp * w.P; i += blockDim.x) {
            const int row = w.m0 + i % w.P;
            if (row < a.lse_seqlen) w.lse_row[int64_t(i / w.P) * a.lse_seqlen + row] = 0.f;
        }
        return false;
    }
    w.qp = (const f16 *)a.q.ptr + base_off(a.q, packed_q, w.b, si.q_start, w.h);
    w.kp = (const f16 *)a.k.ptr + base_off(a.k, packed_k, kb, si.k_start, w.hk);
    w.vp = (const f16 *)a.v.ptr + base_off(a.v, packed_k, kb, si.k_start, w.hk);
    w.op = (f16 *)a.o.ptr + base_off(a.o, packed_q, w.b, si.q_start, w.h);
    w.causal_off = w.sk - w.sq;  // key j visible to query i iff j <= i + causal_off
    int n_end = w.sk;
    if (CAUSAL) n_end = max(0, min(w.sk, w.m0 + w.P + w.causal_off));
    w.n_blocks = (n_end + kFwdBN - 1) / kFwdBN;
    // Negative scales are folded into Q's sign so that the exp argument uses |scale|.
    w.neg = a.softmax_scale < 0.f;
    w.cscale = fabsf(a.softmax_scale) * kLog2e;
    return true;
}

// Narrows w to the rows of 32-row tile t of the workgroup: tile t is head
// w.h + t / (P / 32), positions m0 + 32 (t % (P / 32)) .. + 31.  Returns the
// tile's first position.
__device__ __forceinline__ int fwd_wave(const fa_fwd_args &a, FwdWork &w, int t) {
    const int tiles = w.P >> 5;  // position tiles per head (a power of two)
    const int hp = t >> (31 - __builtin_clz(tiles));
    w.h += hp;
    w.qp += int64_t(hp) * a.q.head_stride;
    w.op += int64_t(hp) * a.o.head_stride;
    w.lse_row += int64_t(hp) * a.lse_seqlen;
    return w.m0 + 32 * (t & (tiles - 1));
}

// Q^T of query qi as B operands: lane (query col, half hh), K step g covers d = 16g + 8hh + 0..7.
template <int HD>
__device__ __forceinline__ void load_q(const fa_fwd_args &a, const FwdWork &w, int qi, int hh, f16x8 (&qB)[HD / 16]) {
#pragma unroll
    for (int g = 0; g < HD / 16; ++g) {
        u32x4 v = zero_u4();
        if (qi < w.sq) v = ldg16(w.qp + int64_t(qi) * a.q.row_stride + 16 * g + 8 * hh);
        if (w.neg) v = neg_h8(v);
        qB[g] = as_h8(v);
    }
}

// Online-softmax state of a wave's 32 queries (this lane's query column).
struct SoftmaxRow {
    float m_t = -INFINITY;  // reference max of scale*log2(e)*S for this lane's query
    float l_p = 0.f;        // partial row sum over this lane half's keys (fp32 P)
};

// One 64-key block of S^T (two 32 x 32 accumulator tiles) -> P^T operands:
// mask (MASK: keys past lim, relative to the block start), running maximum,
// rescale of O, exponentials, row sums.
template <int HD, bool MASK>
__device__ __forceinline__ void softmax_block(f32x16 (&s)[2], f16x8 (&pB)[4], f32x16 (&o)[HD / 32], SoftmaxRow &r,
                                              float cscale, int lim, int hh) {
    if constexpr (MASK) {
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                if (kt * 32 + acc_lrow(e, hh) > lim) s[kt][e] = -INFINITY;
    }
    float mx = s[0][0];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int e = 0; e < 16; ++e) mx = fmaxf(mx, s[kt][e]);
    mx = max_xor32(mx);
    const float mx_t = MASK && mx == -INFINITY ? -INFINITY : mx * cscale;
    if (__builtin_amdgcn_ballot_w64(mx_t > r.m_t) != 0) {
        const float m_new = fmaxf(r.m_t, mx_t);
        const float alpha = m_new == -INFINITY ? 1.f : exp2_fast(r.m_t - m_new);
        r.l_p *= alpha;
#pragma unroll
        for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
            for (int e = 0; e < 16; ++e) o[dt][e] *= alpha;
        r.m_t = m_new;
    }
    const float m_use = r.m_t == -INFINITY ? 0.f : r.m_t;
    float rs = 0.f;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const float x = s[kt][e];
            float p = exp2_fast(fmaf(x, cscale, -m_use));
            if constexpr (MASK) p = x == -INFINITY ? 0.f : p;
            s[kt][e] = p;
            rs += p;
        }
    r.l_p += rs;
#pragma unroll
    for (int gg = 0; gg < 4; ++gg) {
        pB[gg] = pack8(s[gg >> 1], 8 * (gg & 1));
    }
}

// Epilogue: O / l in fp16, LSE = ln(sum exp(scale*S)); empty rows give 0 / 0.
// Dimension tiles [D0, D1); the LSE goes with the first one.
template <int HD, int D0, int D1>
__device__ __forceinline__ void store_row(const fa_fwd_args &a, const FwdWork &w, int qi, int hh,
                                          const f32x16 (&o)[HD / 32], float m_t, float l_tot) {
    if (qi < w.sq) {
        const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
        f16 *orow = w.op + int64_t(qi) * a.o.row_stride;
#pragma unroll
        for (int dt = D0; dt < D1; ++dt)
#pragma unroll
            for (int a4 = 0; a4 < 4; ++a4) {
                f16x4 v;
#pragma unroll
                for (int t = 0; t < 4; ++t) v[t] = (f16)(o[dt][4 * a4 + t] * inv);
                *reinterpret_cast<f16x4 *>(orow + dt * 32 + 8 * a4 + 4 * hh) = v;
            }
        if (D0 == 0 && hh == 0) w.lse_row[qi] = l_tot > 0.f ? (m_t + log2_fast(l_tot)) * kLn2 : 0.f;
    } else if (D0 == 0 && hh == 0 && qi < a.lse_seqlen) {
        w.lse_row[qi] = 0.f;
    }
}

// Splits (fwd_kernel, SPLIT): the workspace starts with an int32 counter per
// workgroup of the unsplit grid (an item: 128 rows), then, 256-byte aligned, the
// items' S x 128 rows' (maximum, sum) and their S x 128 x HD partial O in fp32.
__host__ __device__ __forceinline__ int64_t fwd_count_bytes(int64_t items) { return (items * 4 + 255) & ~int64_t(255); }

// A share's partial result over dimension tiles [D0, D1) of O, in the workspace:
// store() writes share part's, sum() adds all S of an item up in the order of the
// shares, so the sum does not depend on who came last.  Of the n_wgs
// workgroups that have the item's shares, each stores its own and then counts
// itself; the one that counts last finds all of them stored, so none waits for
// another.  live: the lane's row r is a query of the sequence (the others' results
// are not stored).
template <int HD, int D0, int D1>
struct FwdParts {
    static constexpr int N = 8 * (D1 - D0), NT = 512;  // pairs of floats a lane holds, threads
    uint64_t *rows, *pairs;
    __device__ __forceinline__ FwdParts(const fa_fwd_args &a, int64_t items, int item, int S, int thread, int r) {
        rows = reinterpret_cast<uint64_t *>(static_cast<char *>(a.split_ws) + fwd_count_bytes(items));
        pairs = rows + items * S * 128 + int64_t(item) * S * N * NT + thread;
        rows += int64_t(item) * S * 128 + r;
    }
    __device__ __forceinline__ void store(int part, bool live, int hh, const f32x16 (&o)[HD / 32], float m,
                                          float l) const {
        if (!live) return;
        uint64_t *own = pairs + int64_t(part) * N * NT;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const f32x16 &t = o[D0 + i / 8];
            const f32x2 x = {t[2 * (i & 7)], t[2 * (i & 7) + 1]};
            __hip_atomic_store(own + i * NT, __builtin_bit_cast(uint64_t, x), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
        if (D0 == 0 && hh == 0)
            __hip_atomic_store(rows + part * 128, __builtin_bit_cast(uint64_t, f32x2{m, l}), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ __forceinline__ void sum(int S, f32x16 (&o)[HD / 32], float &m, float &l) const {
        auto row_of = [&](int p) {
            return __builtin_bit_cast(f32x2, __hip_atomic_load(rows + p * 128, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        };
        m = -INFINITY;
        l = 0.f;
        for (int p = 0; p < S; ++p) m = fmaxf(m, row_of(p)[0]);
#pragma unroll
        for (int i = D0; i < D1; ++i) o[i] = zero16();
        for (int p = 0; p < S; ++p) {
            const f32x2 ml = row_of(p);
            const float wt = ml[0] == -INFINITY ? 0.f : exp2_fast(ml[0] - m);
            l = fmaf(ml[1], wt, l);
            const uint64_t *slot = pairs + int64_t(p) * N * NT;
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const f32x2 x = __builtin_bit_cast(
                    f32x2, __hip_atomic_load(slot + i * NT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                f32x16 &c = o[D0 + i / 8];
                c[2 * (i & 7)] = fmaf(wt, x[0], c[2 * (i & 7)]);
                c[2 * (i & 7) + 1] = fmaf(wt, x[1], c[2 * (i & 7) + 1]);
            }
        }
    }
};

// Copies of K / V block nb into an LDS tile by all NT threads.  A block that
// runs past the sequence re-reads its last key for the missing rows (masked).
template <int HD, int NT>
struct KvLoader {
    TileCopier<HD, kFwdBN, NT> kcp, vcp;
    __device__ __forceinline__ void init(const fa_fwd_args &a, int wave, int lane) {
        kcp.init(a.k.row_stride, wave, lane);
        vcp.init(a.v.row_stride, wave, lane);
    }
    __device__ __forceinline__ void k(const fa_fwd_args &a, const FwdWork &w, char *smem, uint32_t off, int nb,
                                      int wave, int lane) const {
        const int n0 = nb * kFwdBN;
        if (n0 + kFwdBN <= w.sk)
            kcp.copy_to(lds_addr(smem) + off, w.kp + int64_t(n0) * a.k.row_stride, a.k.row_stride);
        else
            dma_tile<HD, kFwdBN, NT>(smem + off, w.kp, a.k.row_stride, n0, w.sk - 1, wave, lane);
    }
    __device__ __forceinline__ void v(const fa_fwd_args &a, const FwdWork &w, char *smem, uint32_t off, int nb,
                                      int wave, int lane) const {
        const int n0 = nb * kFwdBN;
        if (n0 + kFwdBN <= w.sk)
            vcp.copy_to(lds_addr(smem) + off, w.vp + int64_t(n0) * a.v.row_stride, a.v.row_stride);
        else
            dma_tile<HD, kFwdBN, NT>(smem + off, w.vp, a.v.row_stride, n0, w.sk - 1, wave, lane);
    }
};

// ---------------------------------------------------------------------------
// 4-wave kernel: each wave runs S, softmax and PV of a block in turn; two
// workgroups per CU at head_dim 128 (64 KB LDS, 246 registers), three at
// head_dim 64 (32 KB LDS, at most 168 registers), overlap one wave's softmax
// with the others' MFMAs on each SIMD.  QT = 2 (head_dim 64): each wave takes
// two 32-query tiles of one head and each K / V operand it reads from LDS
// feeds both tiles' MFMAs, which halves the LDS reads per MFMA (at head_dim 64
// a score costs half the MFMA work of head_dim 128 for the same reads of V;
// measured 3-6 % faster at seqlen 8192); two workgroups of 256 queries per
// CU.  The per-tile arithmetic is the same, so the results are the same bits.
// NG = 2: two groups of RW waves (RW = 4: 128 rows, 2: 64 rows) over the same rows
// take the key blocks in turn, each through its own LDS stages, and merge their
// results through LDS at the end.  SPLIT: a query block's key blocks are dealt out to S shares, each
// walked as above, and the shares' results merge through split_ws; L of them, one after another, are
// one workgroup's (1 where the grid then still has a CU for each, so the sum is the same for a GQA
// group packed into a few workgroups and for its expanded heads in many).  A block's place in that
// order depends on its key position alone.
template <int HD, bool CAUSAL, int QT, int NG, int RW, bool SPLIT>
__global__ __launch_bounds__(64 * RW * NG, NG == 2 ? 1 : QT == 2 || HD == 128 ? 2 : 3) void fwd_kernel(
    const fa_fwd_args a, const int num_m_blocks, const int lg, const int S, const int L) {
    constexpr int NT = 256;        // threads that copy a tile together
    constexpr int GT = 64 * RW;    // threads of a wave group
    static_assert(QT == 1 || NG == 1, "two groups: one tile per wave");
    static_assert(NG == 2 || !SPLIT, "splits: two groups");
    static_assert(RW == 4 || (RW == 2 && NG == 2 && !SPLIT), "two row waves: two groups, no splits");
    using C = FwdCfg<HD, NT>;
    constexpr int BM = 32 * RW * QT, BN = C::BN;
    __shared__ __attribute__((aligned(16))) char smem[NG * 2 * C::STAGE];
    __shared__ int ticket;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave8 = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform
    const int wave = NG == 1 ? wave8 : wave8 & (RW - 1), grp = NG == 1 ? 0 : wave8 / RW;
    const int g0 = grp * 2 * C::STAGE;  // the group's LDS stages
    const int hh = lane >> 5;
    FwdWork w;
    const int bp_count = a.batch * (a.nheads >> lg);
    const int unit = SPLIT ? blockIdx.x / bp_count : 0;  // SPLIT: the workgroups of a block of positions in turn
    const int n_wgs = SPLIT ? (S + L - 1) / L : 1;       // ... n_wgs of them
    int part = SPLIT ? unit % n_wgs * L : 0;             // the workgroup's shares: [part, part_end)
    const int part_end = SPLIT ? min(S, part + L) : 1;
    const int bid = SPLIT ? unit / n_wgs * bp_count + (blockIdx.x - unit * bp_count) : blockIdx.x;
    if (!fwd_work<BM, CAUSAL>(a, num_m_blocks, lg, bid, w)) return;

    // The wave's tiles QT * wave + t: one head (the launcher packs at most BM / 64 heads when QT = 2,
    // so a head spans at least 64 positions).
    const int q_lo = fwd_wave(a, w, QT * wave);
    int qi[QT];
    f16x8 qB[QT][HD / 16];
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        qi[t] = q_lo + 32 * t + (lane & 31);
        load_q<HD>(a, w, qi[t], hh, qB[t]);
    }
    wait_vmem();  // only the tile copies are in flight inside the loop

    f32x16 o[QT][HD / 32];
#pragma unroll
    for (int t = 0; t < QT; ++t)
#pragma unroll
        for (int i = 0; i < HD / 32; ++i) o[t][i] = zero16();
    SoftmaxRow row[QT];

    TileReader<HD> rd;
    rd.init(lane);
    KvLoader<HD, NT> ld;
    ld.init(a, RW == 4 ? wave : wave8, lane);
    const int part_step = SPLIT ? S : 1, step = NG * part_step;  // of the workgroup's blocks and of the group's
    int nb0 = part + part_step * grp;                            // the group's first block
    // Copies of the group's block nb into stage st; with two row waves a group,
    // all four waves copy the blocks of both groups.
    auto issue = [&](int nb, int st) FA_INLINE {
        if constexpr (RW == 4) {
            if (nb >= w.n_blocks) return;
            ld.k(a, w, smem, g0 + st * C::STAGE, nb, wave, lane);
            ld.v(a, w, smem, g0 + st * C::STAGE + C::TILE, nb, wave, lane);
        } else {
            const int first = nb - part_step * grp;
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                if (first + part_step * g >= w.n_blocks) return;
                const int off = (2 * g + st) * C::STAGE;
                ld.k(a, w, smem, off, first + part_step * g, wave8, lane);
                ld.v(a, w, smem, off + C::TILE, first + part_step * g, wave8, lane);
            }
        }
    };

    // One key block: S^T = K Q^T, online softmax, O^T += V^T P^T.  MASK is a
    // compile-time switch so the blocks away from the causal diagonal and
    // the sequence end carry no masking work at all.  A tile with no visible
    // key in a block it shares with the wave's other tile gets P = 0 there
    // (its O, sums and maximum unchanged).  The workgroup takes key blocks
    // part, part + S, ... and each of its groups every NG-th of them.
    auto block = [&](int it, auto mask_tag) FA_INLINE {
        constexpr bool MASK = decltype(mask_tag)::value;
        const int buf = it & 1, nb = it * step + nb0;
        wait_vmem();
        __syncthreads();  // block nb is in LDS; every wave is done with stage buf ^ 1
        issue(nb + step, buf ^ 1);
        if (NG > 1 && nb >= w.n_blocks) return;
        const int n0 = nb * BN;
        if (CAUSAL && MASK && n0 > q_lo + 32 * QT - 1 + w.causal_off) return;  // no visible key for this wave
        if (q_lo >= w.sq) return;                                               // no query row of the sequence
        const char *ks = smem + g0 + buf * C::STAGE;
        const char *vs = ks + C::TILE;
        f32x16 s[QT][2];
        f16x8 pB[QT][4];
        auto softmax = [&]() FA_INLINE {
#pragma unroll
            for (int t = 0; t < QT; ++t) {
                const int lim = (CAUSAL ? min(w.sk - 1, qi[t] + w.causal_off) : w.sk - 1) - n0;
                softmax_block<HD, MASK>(s[t], pB[t], o[t], row[t], w.cscale, lim, hh);
            }
        };
        if constexpr (QT == 1) {
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
                s[0][kt] = mfma32(rd.a_operand(ks, 32 * kt, 0), qB[0][0], zero16());
#pragma unroll
                for (int g = 1; g < HD / 16; ++g) s[0][kt] = mfma32(rd.a_operand(ks, 32 * kt, g), qB[0][g], s[0][kt]);
            }
            softmax();
#pragma unroll
            for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
                for (int gg = 0; gg < 4; ++gg) o[0][dt] = mfma32(rd.tr_operand(vs, 16 * gg, dt), pB[0][gg], o[0][dt]);
        } else {
            // Each operand feeds both tiles' MFMAs.  The reads run PIPE steps
            // ahead behind scheduling fences (all of them hoisted to the top
            // would not fit the registers of two waves per SIMD), from the
            // lane's base offsets with this block's stage added once (opaque:
            // hoisted out of the loop, the per-read addresses would hold
            // registers for the whole kernel); each read is one XOR and an
            // immediate (TileReader::a_operand_at).
            constexpr int PIPE = 3, NS = 2 * (HD / 16), NPV = 4 * (HD / 32);
            const int soff = buf * C::STAGE;
            static_assert(C::STAGE % 512 == 0, "stage offsets must be multiples of 512 bytes");
            int ab = rd.a_base + soff, tb0 = rd.tr_base[0] + soff, tb1 = rd.tr_base[1] + soff;
            asm volatile("" : "+v"(ab), "+v"(tb0), "+v"(tb1));
            f16x8 op[PIPE];
            auto rd_k = [&](int u) FA_INLINE {
                op[u % PIPE] = rd.a_operand_at(smem + 32 * (u / (HD / 16)) * (HD * 2), ab, u % (HD / 16));
            };
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < PIPE - 1; ++u) rd_k(u);
#pragma unroll
            for (int u = 0; u < NS; ++u) {
                if (u + PIPE - 1 < NS) rd_k(u + PIPE - 1);
                const int kt = u / (HD / 16), g = u % (HD / 16);
#pragma unroll
                for (int t = 0; t < QT; ++t) s[t][kt] = mfma32(op[u % PIPE], qB[t][g], g == 0 ? zero16() : s[t][kt]);
                __builtin_amdgcn_sched_barrier(0);
            }
            softmax();
            auto rd_v = [&](int u) FA_INLINE {
                op[u % PIPE] = rd.tr_operand_at(smem + C::TILE + 16 * (u & 3) * (HD * 2), tb0, tb1, u >> 2);
            };
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < PIPE - 1; ++u) rd_v(u);
#pragma unroll
            for (int u = 0; u < NPV; ++u) {
                if (u + PIPE - 1 < NPV) rd_v(u + PIPE - 1);
#pragma unroll
                for (int t = 0; t < QT; ++t) o[t][u >> 2] = mfma32(op[u % PIPE], pB[t][u & 3], o[t][u >> 2]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };

    // Blocks [0, n_full) need no mask for any wave of the workgroup: every key
    // is below the sequence end and at or below the diagonal of the first query.
    int n_full = min(w.n_blocks, w.sk / BN);
    if (CAUSAL) n_full = min(n_full, max(0, (w.m0 + w.causal_off + 1) / BN));
    const int64_t items = num_m_blocks * bp_count;  // SPLIT: workgroups of the unsplit grid, and this one's
    const int item = (w.b * (a.nheads >> lg) + (w.h >> lg)) * num_m_blocks + w.m0 / w.P;
    for (;;) {
        // Iterations in which every group has a block, and one without a mask.
        const int last0 = nb0 - part_step * grp + part_step * (NG - 1);  // the last group's first block
        issue(nb0, 0);
        const int it_full = n_full > last0 ? (n_full - 1 - last0) / step + 1 : 0;
        const int n_it = w.n_blocks > part ? (w.n_blocks - 1 - part) / step + 1 : 0;
        for (int it = 0; it < it_full; ++it) block(it, std::false_type{});
        for (int it = it_full; it < n_it; ++it) block(it, std::true_type{});
        if constexpr (NG == 1) {
#pragma unroll
            for (int t = 0; t < QT; ++t)
                store_row<HD, 0, HD / 32>(a, w, qi[t], hh, o[t], row[t].m_t, sum_xor32(row[t].l_p));
        } else {
            // Each group finishes half of the head's dimensions: it hands the other
            // half of its O, and its maxima and sums, to the other group.
            constexpr int H = HD / 64;  // 32-wide dimension tiles of a half
            int t4 = tid & (GT - 1), r = 32 * wave + (lane & 31);
            // SPLIT: opaque to the optimiser, so that the addresses below are formed
            // here and not held through the next share's block loop.
            if constexpr (SPLIT) asm volatile("" : "+v"(t4), "+v"(r));
            const float l_own = sum_xor32(row[0].l_p), m_own = row[0].m_t;
            f32x4 *xo = reinterpret_cast<f32x4 *>(smem);                        // [group][4 H][GT threads]
            f32x2 *xr = reinterpret_cast<f32x2 *>(smem + 2 * 4 * H * GT * 16);  // [group][BM rows]
            __syncthreads();  // every wave is done with the tiles
            if (hh == 0) xr[grp * BM + r] = f32x2{m_own, l_own};
            auto finish = [&](auto grp_tag) FA_INLINE {
                constexpr int GRP = decltype(grp_tag)::value;
#pragma unroll
                for (int i = 0; i < 4 * H; ++i) {
                    const f32x16 &t = o[0][(1 - GRP) * H + i / 4];
                    xo[(GRP * 4 * H + i) * GT + t4] = f32x4{t[4 * (i & 3)], t[4 * (i & 3) + 1], t[4 * (i & 3) + 2],
                                                             t[4 * (i & 3) + 3]};
                }
                __syncthreads();
                const f32x2 other = xr[(1 - GRP) * BM + r];
                float m = fmaxf(m_own, other[0]);
                const float a_own = m_own == -INFINITY ? 0.f : exp2_fast(m_own - m);
                const float a_other = other[0] == -INFINITY ? 0.f : exp2_fast(other[0] - m);
#pragma unroll
                for (int i = 0; i < 4 * H; ++i) {
                    const f32x4 x = xo[((1 - GRP) * 4 * H + i) * GT + t4];
                    f32x16 &t = o[0][GRP * H + i / 4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) t[4 * (i & 3) + e] = fmaf(x[e], a_other, t[4 * (i & 3) + e] * a_own);
                }
                // In group order, so that both groups have the same bits.
                float l = GRP == 0 ? fmaf(other[1], a_other, l_own * a_own) : fmaf(l_own, a_own, other[1] * a_other);
                if constexpr (SPLIT)
                    FwdParts<HD, GRP * H, GRP * H + H>(a, items, item, S, GRP * GT + t4, r)
                        .store(part, qi[0] < w.sq, hh, o[0], m, l);
                else
                    store_row<HD, GRP * H, GRP * H + H>(a, w, qi[0], hh, o[0], m, l);
            };
            if (grp == 0)
                finish(std::integral_constant<int, 0>{});
            else
                finish(std::integral_constant<int, 1>{});
        }
        if (!SPLIT || ++part == part_end) break;
        // The next share, from the start.
        ++nb0;
#pragma unroll
        for (int i = 0; i < HD / 32; ++i) o[0][i] = zero16();
        row[0] = SoftmaxRow();
        __syncthreads();  // every wave has read what the groups exchanged
    }
    if constexpr (SPLIT) {
        wait_vmem();
        __syncthreads();  // every wave's stores have completed
        if (n_wgs > 1) {
            if (tid == 0)
                ticket = __hip_atomic_fetch_add(reinterpret_cast<int32_t *>(a.split_ws) + item, 1, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();
            if (ticket != n_wgs - 1) return;
        }
        auto sum = [&](auto grp_tag) FA_INLINE {
            constexpr int D0 = decltype(grp_tag)::value * (HD / 64), D1 = D0 + HD / 64;
            float m = 0.f, l = 0.f;
            if (qi[0] < w.sq)
                FwdParts<HD, D0, D1>(a, items, item, S, tid, 32 * wave + (lane & 31)).sum(S, o[0], m, l);
            store_row<HD, D0, D1>(a, w, qi[0], hh, o[0], m, l);
        };
        if (grp == 0)
            sum(std::integral_constant<int, 0>{});
        else
            sum(std::integral_constant<int, 1>{});
    }
}

// ---------------------------------------------------------------------------
// Ping-pong kernel: 8 waves over 256 queries.  Waves w and w + 4 share a SIMD
// (waves go to the SIMDs in order, 0..3 then again 0..3); group g = w / 4
// holds 32-query tile 2 (w % 4) + g, so both groups span the workgroup's rows
// and reach the causal diagonal together.  Iteration j (two barriers):
//   group 0: matrix phase [PV of block j - 1, S of block j] | softmax of j
//   group 1: softmax of j - 1 | matrix phase [PV of j - 1, S of j]
// Stage j & 1 holds K_j and V_{j - 1}; the next stage's copies (K_{j + 1},
// V_j) go out at the start of iteration j.  Matrix-phase operands are read
// PIPE steps ahead of their MFMAs with a scheduling fence per step.
constexpr int kPpPipe = 8;

template <int HD, bool CAUSAL>
__global__ __launch_bounds__(512, 1) void fwd_pp_kernel(const fa_fwd_args a, const int num_m_blocks, const int lg) {
    constexpr int NT = 512;
    using C = FwdCfg<HD, NT>;
    constexpr int BM = C::BM, BN = C::BN;
    __shared__ __attribute__((aligned(16))) char smem[2 * C::STAGE];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform
    const int grp = wave >> 2;                                  // 0: matrix phase first
    const int hh = lane >> 5;
    FwdWork w;
    if (!fwd_work<BM, CAUSAL>(a, num_m_blocks, lg, blockIdx.x, w)) return;

    const int q_lo = fwd_wave(a, w, 2 * (wave & 3) + grp);
    const int qi = q_lo + (lane & 31);
    f16x8 qB[HD / 16];
    load_q<HD>(a, w, qi, hh, qB);
    wait_vmem();  // only the tile copies are in flight inside the loop

    f32x16 o[HD / 32];
#pragma unroll
    for (int i = 0; i < HD / 32; ++i) o[i] = zero16();
    SoftmaxRow row;

    TileReader<HD> rd;
    rd.init(lane);
    KvLoader<HD, NT> ld;
    ld.init(a, wave, lane);

    // Last key this wave sees; blocks [0, nbw) hold its keys, and blocks
    // [0, n_full) need no mask for any of its queries.
    const int wave_last_key = CAUSAL ? min(w.sk - 1, q_lo + 31 + w.causal_off) : w.sk - 1;
    const int nbw = q_lo < w.sq ? max(0, min(w.n_blocks, (wave_last_key + BN) / BN)) : 0;
    int n_full = min(w.n_blocks, w.sk / BN);
    if (CAUSAL) n_full = min(n_full, max(0, (q_lo + w.causal_off + 1) / BN));

    f32x16 s[2];
    f16x8 pB[4];
    // Matrix phase of iteration j: O^T += V_{j-1}^T P_{j-1}^T (DO_PV), then
    // S_j^T = K_j Q^T (DO_S); step t < NPV is a PV MFMA, the rest S MFMAs.
    constexpr int NPV = 4 * (HD / 32), NS = 2 * (HD / 16);
    auto matrix = [&](int j, auto pv_tag, auto s_tag) FA_INLINE {
        constexpr bool DO_PV = decltype(pv_tag)::value, DO_S = decltype(s_tag)::value;
        constexpr int T0 = DO_PV ? 0 : NPV, T1 = DO_S ? NPV + NS : NPV;
        // The lane's read bases with stage j & 1 added once (opaque: hoisted out
        // of the loop, the per-read addresses would hold registers for the
        // whole kernel); each read is then one XOR and an immediate
        // (TileReader::a_operand_at).
        const int soff = (j & 1) * C::STAGE;
        static_assert(C::STAGE % 512 == 0, "stage offsets must be multiples of 512 bytes");
        int ab = rd.a_base + soff, tb0 = rd.tr_base[0] + soff, tb1 = rd.tr_base[1] + soff;
        asm volatile("" : "+v"(ab), "+v"(tb0), "+v"(tb1));
        f16x8 opnd[kPpPipe];
        auto read = [&](int t) FA_INLINE {
            if (t < NPV)
                opnd[t % kPpPipe] = rd.tr_operand_at(smem + C::TILE + 16 * (t & 3) * (HD * 2), tb0, tb1, t >> 2);
            else
                opnd[t % kPpPipe] =
                    rd.a_operand_at(smem + 32 * ((t - NPV) / (HD / 16)) * (HD * 2), ab, (t - NPV) % (HD / 16));
        };
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = T0; t < T0 + kPpPipe - 1 && t < T1; ++t) read(t);
#pragma unroll
        for (int t = T0; t < T1; ++t) {
            if (t + kPpPipe - 1 < T1) read(t + kPpPipe - 1);
            if (t < NPV) {
                o[t >> 2] = mfma32(opnd[t % kPpPipe], pB[t & 3], o[t >> 2]);
            } else {
                const int u = t - NPV, kt = u / (HD / 16), g = u % (HD / 16);
                s[kt] = mfma32(opnd[t % kPpPipe], qB[g], g == 0 ? zero16() : s[kt]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto softmax = [&](int j, auto mask_tag) FA_INLINE {
        constexpr bool MASK = decltype(mask_tag)::value;
        const int lim = (CAUSAL ? min(w.sk - 1, qi + w.causal_off) : w.sk - 1) - j * BN;
        softmax_block<HD, MASK>(s, pB, o, row, w.cscale, lim, hh);
    };
    auto softmax_any = [&](int j) FA_INLINE {
        if (j < n_full)
            softmax(j, std::false_type{});
        else
            softmax(j, std::true_type{});
    };
    // Start of iteration j: K_j and V_{j-1} are in stage j & 1 (every wave's
    // copies have landed) and stage (j + 1) & 1 is free: the next copies go out.
    auto top = [&](int j) FA_INLINE {
        wait_vmem();
        __syncthreads();
        if (j < w.n_blocks) {
            if (j + 1 < w.n_blocks) ld.k(a, w, smem, ((j + 1) & 1) * C::STAGE, j + 1, wave, lane);
            ld.v(a, w, smem, ((j + 1) & 1) * C::STAGE + C::TILE, j, wave, lane);
        }
    };
    auto mid = []() FA_INLINE { __builtin_amdgcn_s_barrier(); };
    using T = std::true_type;
    using F = std::false_type;

    // Every wave runs iterations 0..n_blocks (two barriers each); a wave does
    // S for blocks j < nbw and PV for 1 <= j <= nbw.
    if (w.n_blocks > 0) ld.k(a, w, smem, 0, 0, wave, lane);
    int j = 1;
    if (grp == 0) {
        top(0);
        if (nbw > 0) matrix(0, F{}, T{});
        mid();
        if (nbw > 0) softmax_any(0);
        for (; j < min(nbw, n_full); ++j) {
            top(j);
            matrix(j, T{}, T{});
            mid();
            softmax(j, F{});
        }
        for (; j < nbw; ++j) {
            top(j);
            matrix(j, T{}, T{});
            mid();
            softmax(j, T{});
        }
        if (nbw > 0) {
            top(nbw);
            matrix(nbw, T{}, F{});
            mid();
            j = nbw + 1;
        }
    } else {
        top(0);
        mid();
        if (nbw > 0) matrix(0, F{}, T{});
        for (; j < min(nbw, n_full + 1); ++j) {
            top(j);
            softmax(j - 1, F{});
            mid();
            matrix(j, T{}, T{});
        }
        for (; j < nbw; ++j) {
            top(j);
            softmax(j - 1, T{});
            mid();
            matrix(j, T{}, T{});
        }
        if (nbw > 0) {
            top(nbw);
            softmax_any(nbw - 1);
            mid();
            matrix(nbw, T{}, F{});
            j = nbw + 1;
        }
    }
    for (; j <= w.n_blocks; ++j) {
        top(j);
        mid();
    }
    store_row<HD, 0, HD / 32>(a, w, qi, hh, o, row.m_t, sum_xor32(row.l_p));
}

// Varlen work order (order_items in fa_common.h): item it = b * nmb + mb is
// block mb of P query positions of sequence b, its work about positions x
// keys seen by the block's last position, in buckets of P x 64; blocks past a
// sequence's end come last (they still write LSE padding).
// Workgroups past the first zero the output rows of no sequence (order_wgs is 0
// without a work_order).
__global__ __launch_bounds__(kOrderThreads) void fwd_order_kernel(const fa_fwd_args a, const int nmb, const int P,
                                                                  const int order_wgs) {
    if (int(blockIdx.x) >= order_wgs) {
        zero_gaps(a.o, a.cu_seqlens_q, a.batch, a.lse_seqlen, a.o_rows, a.nheads, a.head_dim, blockIdx.x - order_wgs,
                  gridDim.x - order_wgs);
        return;
    }
    order_items(a.batch * nmb, [&](int it) {
        const int b = it / nmb, mb = it - b * nmb;
        const int sq = a.cu_seqlens_q[b + 1] - a.cu_seqlens_q[b];
        const int sk = a.cu_seqlens_k ? a.cu_seqlens_k[b + 1] - a.cu_seqlens_k[b] : a.seqlen_k;
        const int m0 = mb * P;
        if (m0 >= sq) return -1;
        const int64_t rows = min(P, sq - m0);
        const int64_t keys = a.causal ? max(0, min(sk, m0 + P + sk - sq)) : max(sk, 0);
        return int(min<int64_t>(rows * keys / (int64_t(P) * 64), kOrderBuckets - 1));
    }, a.work_order, true);
}

static int launch_order(const fa_fwd_args &a, int nmb, int P, hipStream_t stream) {
    if (!a.cu_seqlens_q || (!a.work_order && a.o_rows <= 0)) return FA_OK;
    const int order_wgs = a.work_order ? 1 : 0;
    hipLaunchKernelGGL(fwd_order_kernel, dim3(order_wgs + (a.o_rows > 0 ? kZeroBlocks : 0)), dim3(kOrderThreads), 0,
                       stream, a, nmb, P, order_wgs);
    return int(hipGetLastError());
}

// log2 of the query heads per workgroup for a BM-row kernel: the largest
// power of two that divides the GQA group (those heads read the same K / V)
// and leaves whole 32-row tiles per head.  The K / V tiles a workgroup loads
// then serve gp heads instead of one, and the workgroup spans BM / gp
// positions, so a causal block wastes less on the diagonal.
static int fwd_pack_log2(const fa_fwd_args &a, int BM) {
    const int group = a.nheads / a.nheads_k;
    int lg = 0;
    while ((64 << lg) <= BM && group % (2 << lg) == 0) ++lg;
    return lg;
}

// Causal calls whose longest row sees at most twice the average row's keys or so
// (queries over at most as many earlier keys again), and those of a square.
static bool causal_near(const fa_fwd_args &a) { return a.causal && a.seqlen_k <= 2 * int64_t(a.seqlen_q); }
static bool causal_square(const fa_fwd_args &a) {
    return a.causal && 10 * int64_t(a.seqlen_k) <= 11 * int64_t(a.seqlen_q);
}

// How the keys of a query block are shared: wave groups per workgroup and shares
// (splits) per query block.  A group rounds P to fp16 against its own running
// maximum, so a row's bits depend on this plan, and with it on batch, heads and
// lengths.  They must not depend on how many heads share a workgroup (a GQA group
// gives the bits of its expanded heads), so the rules count work that packing does
// not change: W, 128-row blocks in 32-row tiles (what the packed heads of short
// calls fill), and the 128- and 64-row blocks of unpacked heads (U, U64), the most
// workgroups that any form of the call launches.  NB: key blocks of the longest row.
// Measured on MI355X, us at one group of 4 row waves -> as planned (row waves x
// groups x splits), head_dim 128 unless noted:
//   one workgroup per CU leaves each SIMD one wave; a second group halves the
//   chain of key blocks (1.82 us for a pair of blocks against 2 x 1.22):
//     b1 s1024 32/8 causal (W 256): 28.3 -> 25.7 (4 x 2 x 1)   s2048 16/16: 45.7 -> 38.3
//     b1 s4096 16/16 causal (W 512): 110 -> 93                 1024 x 16384 keys 32/8: 328 -> 294
//   a workgroup of two groups has a CU to itself, so it loses where one-group ones
//   would share CUs: without a causal square (W 512, s4096 no mask: 153 -> 159;
//   256 x 4000 keys: 177 -> 208; 1024 x 2048 causal: 69 -> 72), past W 512 (W 768,
//   s2048: 74.5 -> 82) and for unpacked heads of few queries (b16 32/32, 64 x 1300:
//   69 -> 77; b32 16/16, 16 x 1400: 69 -> 75); and on short chains (W 256, s256:
//   11.8 -> 12.3; one block: 5.0 -> 5.5);
//   with CUs still idle and long chains, splits take them (one launch to clear the
//   counters and a merge: about 8 us, 2 more per split):
//     512 rows x 16384 keys 32/8: 311 -> 160 (4 x 2 x 2)       128 rows: 309 -> 60 (4 x 2 x 8)
//     512 x 8192 16/4 d64: 127 -> 38 (4 x 2 x 4)
//   and where heads do not pack, their workgroups walk the same shares in turn: 16
//     queries x 8000 keys b8: 32/8 159 -> 61 (4 x 2 x 4), 32/32 188 -> 200
struct FwdPlan {
    int groups, splits;
};
static FwdPlan fwd_plan(const fa_fwd_args &a) {
    const int64_t heads = int64_t(a.batch) * a.nheads, len = a.lse_seqlen, cus = device_cus();
    const int64_t W = (heads * ((len + 31) / 32) + 3) / 4, U = heads * ((len + 127) / 128), U64 = heads * ((len + 63) / 64);
    const int NB = (a.seqlen_k + kFwdBN - 1) / kFwdBN;
    const bool half = 2 * W <= cus;  // half of the CUs would idle
    // The least key blocks for two groups (64-row blocks, fwd_narrow, pay from 2 on).
    const int least = half                ? !a.cu_seqlens_q && U64 <= cus ? 2 : 8
                      : a.head_dim == 64 ? (causal_near(a) ? 6 : 8)
                                         : (causal_near(a) ? 9 : 12);
    const bool few = 2 * U <= 3 * cus, dense = !a.cu_seqlens_q;  // varlen: the work order lists unsplit blocks
    FwdPlan plan = {1, 1};
    if (W > cus)
        plan.groups = W <= 2 * cus && causal_square(a) && NB >= 32 ? 2 : 1;
    else if (few || (half && dense && U <= 2 * cus))
        plan.groups = NB >= least ? 2 : 1;
    if (!half || plan.groups == 1 || !dense) return plan;
    const double pairs = 0.5 * NB, unit = a.head_dim == 128 ? 1.84 : 1.31;
    const double unsplit = pairs * (a.head_dim == 128 ? 1.58 : 0.9), one_group = pairs * 2.44;
    double best = unsplit;
    for (int S = 2; S <= 16 && W * S <= cus; ++S) {
        const double t = pairs / S * unit + 6 + 2 * S;
        if (t < best) {
            best = t;
            plan.splits = S;
        }
    }
    // Where the unpacked form of the call fills the chip by itself, it gains nothing
    // by two groups or shares and takes the shares one after another (5 - 18 % slower,
    // the more the shorter): only where the packed form gains much.  16 queries of b16
    // 32/8 and 32/32 heads, us in one group -> as planned: 3000 keys 66 -> 46 and 137 ->
    // 154, 20000 keys 392 -> 261 and (10000) 439 -> 465; head_dim 64, 8000 keys, where
    // two groups do without shares: 122 -> 84 and 184 -> 194.
    if (!few && a.head_dim == 64) plan.splits = 1;
    if (!few && a.head_dim == 128 && best > 0.6 * one_group) plan = {1, 1};
    if (few && U >= cus && best > 0.55 * unsplit) plan.splits = 1;
    return plan;
}
// Workgroups of the unsplit grid of BM-row blocks.
static int64_t fwd_items(const fa_fwd_args &a, int BM) {
    const int lg = fwd_pack_log2(a, BM), P = BM >> lg;
    return int64_t((a.lse_seqlen + P - 1) / P) * a.batch * (a.nheads >> lg);
}
static size_t fwd_split_bytes(const fa_fwd_args &a, int S) {
    const int64_t items = fwd_items(a, 128);
    return S > 1 ? size_t(fwd_count_bytes(items) + items * S * 128 * (8 + 4 * int64_t(a.head_dim))) : 0;
}

// Whether the two wave groups of an unsplit dense call have 2 row waves each
// (64-row blocks) instead of 4: the same bits, read half as much LDS a workgroup
// (1.58 us a pair of blocks against 1.82; 0.9 against 1.31 at head_dim 64), so they
// win where their grid still has a CU for each workgroup, and a little past that
// where a causal square's later workgroups are short.  Measured on MI355X, us in
// 128-row -> 64-row blocks (workgroups of the latter), head_dim 128 unless noted:
//   b1 s509 32/8 causal (256): 15.4 -> 13.5       b1 s1024 16/2 causal (256): 23.7 -> 21.3
//   b1 s1200 16/2 causal (304): 26.7 -> 25.1      b1 s700 32/8 causal (352): 18.6 -> 18.1
//   b2 s350 32/8 causal (352): 14.5 -> 16.6       700 x 1050 keys causal (352): 26.3 -> 29.9
//   b1 s2048 8/8 causal (512): 41.8 -> 44.8       b4 200 x 8000 keys 32/4 (448): 144 -> 237
//   d64 b2 s2048 8/8 causal (512): 29.7 -> 26.7   d64 1024 x 2048 keys causal (512): 30.6 -> 29.9
//   d64 2048 x 6144 keys causal (512): 77 -> 79   d64 256 x 1024 keys no mask (384): 18.0 -> 19.1
static bool fwd_narrow(const fa_fwd_args &a) {
    const int64_t n = fwd_items(a, 64), cus = device_cus();
    if (n <= cus) return true;
    if (a.head_dim == 64) return n <= 2 * cus && causal_near(a);
    return 2 * n <= 3 * cus && causal_square(a) && a.seqlen_k > 9 * kFwdBN;
}

template <int HD, bool CAUSAL>
static int launch_fwd(const fa_fwd_args &a, hipStream_t stream) {
    // The ping-pong kernel when its grid fills the chip at least twice over
    // and sequences reach 2048 rows; the 4-wave kernel otherwise (and at
    // head_dim 64, where it measured faster).  Below 2048 rows the 128-row
    // blocks waste less on causal diagonals and ragged sequence ends and deal
    // out more evenly (measured varlen causal, 32 / 8 heads: 64 x 1024 rows
    // +3 %, 64 x U[64, 1024] +14 %; 32 x 2048 even; 16 x 4096 -5 %).  Both
    // give the bits of one wave group, and so does the two-tile kernel below;
    // where the plan has two, neither is taken, however large the grid is that the
    // unpacked heads make.
    const FwdPlan plan = fwd_plan(a);
    if constexpr (HD == 128) {
        constexpr int BM = FwdCfg<HD, 512>::BM;
        const int lg = fwd_pack_log2(a, BM), P = BM >> lg;
        const int64_t pp_m_blocks = (a.lse_seqlen + P - 1) / P;
        const int64_t pp_grid = pp_m_blocks * a.batch * (a.nheads >> lg);
        if (plan.groups == 1 && pp_grid >= 2 * int64_t(device_cus()) && a.lse_seqlen >= 2048) {
            if (pp_grid > 0x7fffffff) return FA_ERR_INVALID_ARG;
            const int rc = launch_order(a, int(pp_m_blocks), P, stream);
            if (rc) return rc;
            hipLaunchKernelGGL((fwd_pp_kernel<HD, CAUSAL>), dim3(unsigned(pp_grid)), dim3(512), 0, stream, a,
                               int(pp_m_blocks), lg);
            return int(hipGetLastError());
        }
    }
    // Head_dim 64: two query tiles per wave when that grid still fills the chip
    // twice over.  A wave's two tiles must be one head's, so at most 4 heads
    // share a workgroup (64 positions each).
    if constexpr (HD == 64) {
        constexpr int BM2 = 2 * FwdCfg<HD, 256>::BM;
        const int lg = min(fwd_pack_log2(a, BM2), 2), P = BM2 >> lg;
        const int64_t m_blocks = (a.lse_seqlen + P - 1) / P;
        const int64_t grid = m_blocks * a.batch * (a.nheads >> lg);
        if (plan.groups == 1 && grid >= 2 * int64_t(device_cus())) {
            if (grid > 0x7fffffff) return FA_ERR_INVALID_ARG;
            const int rc = launch_order(a, int(m_blocks), P, stream);
            if (rc) return rc;
            hipLaunchKernelGGL((fwd_kernel<HD, CAUSAL, 2, 1, 4, false>), dim3(unsigned(grid)), dim3(256), 0, stream, a,
                               int(m_blocks), lg, 1, 1);
            return int(hipGetLastError());
        }
    }
    const int S = a.split_ws && a.split_ws_bytes >= int64_t(fwd_split_bytes(a, plan.splits)) ? plan.splits : 1;
    if (plan.groups == 2 && S == 1 && !a.cu_seqlens_q && fwd_narrow(a)) {
        const int lg = fwd_pack_log2(a, 64), P = 64 >> lg;
        const int m_blocks = (a.lse_seqlen + P - 1) / P;
        const int64_t grid = int64_t(m_blocks) * a.batch * (a.nheads >> lg);
        if (grid > 0x7fffffff) return FA_ERR_INVALID_ARG;
        if (grid == 0) return FA_OK;
        hipLaunchKernelGGL((fwd_kernel<HD, CAUSAL, 1, 2, 2, false>), dim3(unsigned(grid)), dim3(256), 0, stream, a,
                           m_blocks, lg, 1, 1);
        return int(hipGetLastError());
    }
    constexpr int BM = FwdCfg<HD, 256>::BM;
    const int lg = fwd_pack_log2(a, BM), P = BM >> lg;
    const int num_m_blocks = (a.lse_seqlen + P - 1) / P;
    const int64_t grid = int64_t(num_m_blocks) * a.batch * (a.nheads >> lg);
    if (grid > 0x7fffffff) return FA_ERR_INVALID_ARG;
    const int rc = launch_order(a, num_m_blocks, P, stream);
    if (rc || grid == 0) return rc;
    // Shares that a workgroup takes one after another: few enough workgroups for
    // one CU each (b32 8/8, 2 x 8000 keys, 256 blocks x 4 shares: 240 us in 1024
    // workgroups, 216 in 256, 189 without shares).
    int L = 1;
    while (L < S && grid * ((S + L - 1) / L) > device_cus()) ++L;
    if (L < S) {  // several workgroups a block: they count
        const int rc2 = clear_counts(a.split_ws, grid, stream);
        if (rc2) return rc2;
    }
    auto go = [&](auto ng_tag, auto split_tag) {
        constexpr int NG = decltype(ng_tag)::value;
        hipLaunchKernelGGL((fwd_kernel<HD, CAUSAL, 1, NG, 4, decltype(split_tag)::value>),
                           dim3(unsigned(grid * ((S + L - 1) / L))), dim3(256 * NG), 0, stream, a, num_m_blocks, lg, S, L);
    };
    using G1 = std::integral_constant<int, 1>;
    using G2 = std::integral_constant<int, 2>;
    if (S > 1)
        go(G2{}, std::true_type{});
    else
        plan.groups == 2 ? go(G2{}, std::false_type{}) : go(G1{}, std::false_type{});
    return int(hipGetLastError());
}

}  // namespace fa

extern "C" int fa_fwd(const fa_fwd_args *args, void *stream) {
    if (!args) return FA_ERR_INVALID_ARG;
    const fa_fwd_args &a = *args;
    if (a.head_dim != 64 && a.head_dim != 128) return FA_ERR_UNSUPPORTED;
    if (a.batch < 0 || a.seqlen_q < 0 || a.seqlen_k < 0 || a.nheads <= 0 || a.nheads_k <= 0 ||
        a.nheads % a.nheads_k != 0 || !a.lse || a.lse_seqlen < a.seqlen_q || !fa::split_ws_aligned(a.split_ws))
        return FA_ERR_INVALID_ARG;
    if (fa::check_tensor(a.q, true) || fa::check_tensor(a.k, true) || fa::check_tensor(a.v, true) ||
        fa::check_tensor(a.o, true))
        return FA_ERR_INVALID_ARG;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (a.head_dim == 128)
        return a.causal ? fa::launch_fwd<128, true>(a, s) : fa::launch_fwd<128, false>(a, s);
    return a.causal ? fa::launch_fwd<64, true>(a, s) : fa::launch_fwd<64, false>(a, s);
}

extern "C" size_t fa_fwd_split_bytes(const fa_fwd_args *a) {
    if (!a || a->batch <= 0 || a->seqlen_q <= 0 || a->seqlen_k <= 0 || a->nheads <= 0 || a->nheads_k <= 0 ||
        (a->head_dim != 64 && a->head_dim != 128))
        return 0;
    return fa::fwd_split_bytes(*a, fa::fwd_plan(*a).splits);
}

extern "C" size_t fa_fwd_order_len(const fa_fwd_args *a) {
    if (!a || a->batch <= 0 || a->lse_seqlen <= 0) return 0;
    return size_t(a->batch) * size_t((a->lse_seqlen + 31) / 32);  // blocks of 32 positions at the least
}
