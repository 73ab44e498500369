// Attention kernels for short contexts (documents of a few hundred tokens, small batches), forward and backward.
//
// The tiled kernels give a workgroup 128 - 256 rows and walk its keys (queries) in one chain of barriers; with short documents that
// chain is most of the launch, its workgroups leave compute units idle, and 256 rows span several documents.  Here a workgroup of
// four (two: mi_attn_short_pairs) wavefronts owns 32 rows, and the wavefronts split the other axis: wavefront w takes tiles w, w + 4 (w + 2), ... of 32
// tokens, each through its own LDS stages with direct global -> LDS loads and no barrier, and the partial results meet in
// LDS at the end, in a fixed order.  A document of 512 tokens is a chain of at most four (eight) tiles.  The mask interval of a row comes from one
// load of the cumulative lengths and a search in registers.
// The price is operand traffic: a tile serves 32 rows instead of 128 or 256, so long contexts stay with the tiled kernels
// (see mi_attn_fwd_is_short and mi_attn_bwd_short).
#pragma once
#include "attn_common.h"

namespace {

constexpr int kShortRows = 32;

// Largest j < n_docs with cu[j] <= t and the bounds of that document on both axes, as find_doc gives them; for up to 63 documents the
// lengths sit one per lane.
struct DocBounds { int qs, qe, ks, ke; };
template <bool KEY>
__device__ __forceinline__ DocBounds short_doc(const AttnParams& p, int t, int lane) {
    DocBounds d;
    if (p.n_docs == 1) {
        d.qs = p.cu_q[0]; d.qe = p.cu_q[1]; d.ks = p.cu_k[0]; d.ke = p.cu_k[1];
    } else if (p.n_docs <= 63) {
        const int at = lane < p.n_docs ? lane : p.n_docs;
        const int cq = p.cu_q[at], ck = p.cu_k[at];
        const int c = KEY ? ck : cq;
        int j = 0;
#pragma unroll
        for (int step = 32; step > 0; step >>= 1) {
            const int mid = j + step, v = __shfl(c, mid & 63, MI_WAVE);
            if (mid < p.n_docs && v <= t) j = mid;
        }
        d.qs = __shfl(cq, j, MI_WAVE); d.qe = __shfl(cq, j + 1, MI_WAVE);
        d.ks = __shfl(ck, j, MI_WAVE); d.ke = __shfl(ck, j + 1, MI_WAVE);
    } else {
        const int j = find_doc(KEY ? p.cu_k : p.cu_q, p.n_docs, t);
        d.qs = p.cu_q[j]; d.qe = p.cu_q[j + 1]; d.ks = p.cu_k[j]; d.ke = p.cu_k[j + 1];
    }
    return d;
}
// key_range / query_range of attn_common.h
__device__ __forceinline__ void short_key_range(const AttnParams& p, int t, int lane, int& klo, int& khi) {
    const DocBounds d = short_doc<false>(p, t, lane);
    klo = d.ks;
    khi = p.causal ? min(d.ks + (t - d.qs) + (d.ke - d.ks) - (d.qe - d.qs) + 1, d.ke) : d.ke;
    if (t >= p.total_q) klo = khi = 0;
    if (khi < klo) khi = klo;
}
__device__ __forceinline__ void short_query_range(const AttnParams& p, int u, int lane, int& qlo, int& qhi) {
    const DocBounds d = short_doc<true>(p, u, lane);
    qhi = d.qe;
    qlo = p.causal ? max(d.qs + (u - d.ks) - ((d.ke - d.ks) - (d.qe - d.qs)), d.qs) : d.qs;
    if (u >= p.total_k) qlo = qhi = 0;
    if (qlo > qhi) qlo = qhi;
}
// union of the wavefront's intervals, from a multiple of 32 on
__device__ __forceinline__ void short_tiles(int lo, int hi, int& wmin, int& wmax, int& t0, int& n_tiles) {
    wmin = group_min<64>(hi > lo ? lo : 0x7fffffff);
    wmax = group_max<64>(hi > lo ? hi : 0);
    // the same in every lane; made scalar, as loop control and the base address of a direct load have to be
    const bool any = wmax > wmin;
    t0 = __builtin_amdgcn_readfirstlane(any ? wmin & ~31 : 0);
    n_tiles = __builtin_amdgcn_readfirstlane(any ? (wmax - t0 + 31) / 32 : 0);
}

// One wavefront's two (three) tiles of 32 tokens, in STAGES stages.  The chains are short, so what hides the loads is the other workgroups of the
// compute unit: one stage (8192 tokens x 32 heads of 128 in documents of 512: forward 240 us with two, 137 with one), except for dK / dV
// of 96 and 128 features, whose registers leave room for one workgroup anyway.
template <int D, int WAVES, int STAGES = 1, int TILES = 2> struct ShortStages {
    using Tile = LdsTile<D>;
    static constexpr int kTile = 32 * Tile::RB, kLoads = Tile::kInstrs / 2;
    static constexpr int kBytes = TILES * STAGES * kTile;
    static constexpr int kSmem = WAVES * kBytes;
    char* base;
    __device__ __forceinline__ char* first(int buf = 0) const { return base + buf * TILES * kTile; }
    __device__ __forceinline__ char* second(int buf = 0) const { return base + buf * TILES * kTile + kTile; }
    __device__ __forceinline__ char* third(int buf = 0) const { return base + buf * TILES * kTile + 2 * kTile; }
    // Before a stage is loaded again its reads must have returned.
    static __device__ __forceinline__ void reads_done() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
};

template <int D, int WAVES> constexpr int kShortRed = WAVES * 16 * (D / 32) * 64 * 4;      // an accumulator set of every wavefront
// Sums over the wavefronts meet in LDS ([wave][16 DT][64] floats); then each of them takes 4 / WAVES of the quads of every feature tile (rows 8 a + 4 g + c).
template <int D> __device__ __forceinline__ void short_store(float* red, int wave, int lane, const f32x16_t (&acc)[D / 32]) {
    float* mine = red + wave * (16 * (D / 32) * 64) + lane;
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) mine[(dt * 16 + r) * 64] = acc[dt][r];
}
template <int D, int WAVES> __device__ __forceinline__ void short_sums(const float* red, int wave, int lane, float (&x)[4 / WAVES][D / 32][4]) {
    constexpr int kSet = 16 * (D / 32) * 64;
#pragma unroll
    for (int j = 0; j < 4 / WAVES; ++j)
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float* at = red + (dt * 16 + 4 * (wave * (4 / WAVES) + j) + c) * 64 + lane;
                if constexpr (WAVES == 4) x[j][dt][c] = (at[0] + at[kSet]) + (at[2 * kSet] + at[3 * kSet]);
                else x[j][dt][c] = at[0] + at[kSet];
            }
}
// Rotation by minus the position's angles of features 32 dt + 8 a + 4 g + c (see unrotate_acc)
template <int D> __device__ __forceinline__ void short_unrotate(float (&x)[D / 32][4], const AttnParams& p, int64_t pos, int a, int g) {
    constexpr int DT = D / 32;
    pos = pos < 0 ? 0 : (pos >= p.table_rows ? p.table_rows - 1 : pos);
    if (p.unrotate == 1) {
        const elem_t* cr = p.cos + pos * D + 8 * a + 4 * g;
        const elem_t* sr = p.sin + pos * D + 8 * a + 4 * g;
#pragma unroll
        for (int dt = 0; dt < DT / 2; ++dt) {
            const uint2 cw = *reinterpret_cast<const uint2*>(cr + 32 * dt), sw = *reinterpret_cast<const uint2*>(sr + 32 * dt);
            const float c4[4] = {elem_lo(cw.x), elem_hi(cw.x), elem_lo(cw.y), elem_hi(cw.y)};
            const float s4[4] = {elem_lo(sw.x), elem_hi(sw.x), elem_lo(sw.y), elem_hi(sw.y)};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float x0 = x[dt][c], x1 = x[dt + DT / 2][c];
                x[dt][c] = x0 * c4[c] + x1 * s4[c];
                x[dt + DT / 2][c] = x1 * c4[c] - x0 * s4[c];
            }
        }
    } else {
        const float* cr = p.cos32 + pos * (D / 2) + 4 * a + 2 * g;
        const float* sr = p.sin32 + pos * (D / 2) + 4 * a + 2 * g;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            const float2 c2 = *reinterpret_cast<const float2*>(cr + 16 * dt), s2 = *reinterpret_cast<const float2*>(sr + 16 * dt);
            rotate_complex_pair(x[dt][0], x[dt][1], c2.x, -s2.x);
            rotate_complex_pair(x[dt][2], x[dt][3], c2.y, -s2.y);
        }
    }
}
template <int D> __device__ __forceinline__ void short_write(elem_t* row, const float (&x)[D / 32][4], float scale) {
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
        *reinterpret_cast<uint2*>(row + 32 * dt) = make_uint2(pack_elem2(x[dt][0] * scale, x[dt][1] * scale), pack_elem2(x[dt][2] * scale, x[dt][3] * scale));
}

// Host side: two wavefronts to a block instead of four.  What comes before and after a chain of tiles costs every wavefront of a block alike, and of four the short
// chains of packed documents leave some without a tile; so two do a block in half as many turns of the chip again, as long as there are blocks
// enough for it to wait for all of them and not for the longest chain.  That is twice as long now, and its length is not known here, only
// the mean: hence enough heads, so that one document of half the tokens among 16 small ones is level too (8 heads of 64: 1.25 forward, 1.28
// backward).  Two / four, over 691 calls of 4 - 32 heads of 32 - 128, 1024 - 16384 tokens, documents ragged, whole, with a long tail and with one long one among
// short ones: forward .67 - 1.02, mean .85, backward .65 - 1.03, mean .79, where the rule takes two.  us: 16 heads of 64, 4096 tokens, documents of 20 - 380:
// here four / two: backward 50.3 / 38.4; 32 heads: 92.2 / 68.5, forward 30.2 / 24.2; 16 heads of 128 35.0 / 25.4.
// `blocks`: of 32 rows, of both kinds in a backward pass
static inline bool mi_attn_short_pairs(const mi_attn_args* a, bool backward, int64_t blocks) {
    const int64_t rows = a->total_q > a->total_k ? a->total_q : a->total_k, units = mi_compute_units(), d = a->head_dim;
    if (a->n_docs <= 1) return false;
    const int64_t chain = (a->causal ? 1 : 2) * rows / a->n_docs;
    if (backward)
        return d <= 64 && a->n_q_heads == a->n_kv_heads && a->n_q_heads >= 12 && blocks >= (d == 64 ? 6 : 7) * units && blocks * (d == 64 ? 64 : 40) >= chain * units;
    if (d <= 64) return a->n_q_heads >= 24 && blocks >= 4 * units && blocks * (d == 64 ? 56 : 28) >= chain * units;
    return a->n_q_heads >= 16 && blocks >= (a->n_q_heads >= 24 ? 4 : 5) * units && blocks * 96 >= chain * units;
}

static inline int64_t mi_attn_short_blocks(const mi_attn_args* a, int64_t heads) {
    const int64_t rows = a->total_q > a->total_k ? a->total_q : a->total_k;
    return (rows + kShortRows - 1) / kShortRows * heads;
}

// Whether a forward pass goes to these kernels, by its workgroups of 32 rows (rows / 32 x query heads).  A compute unit holds eight of
// them up to 64 features, two above.  The tiled kernels wait for the longest chain of a workgroup, which is what these kernels shorten; they
// gain where that chain runs alone: few workgroups, and causal documents, whose last rows have twice the average work.  They lose where the
// tiled kernels have work for every compute unit all along.  Short / tiled, at 512 | 1024 | 1536 | 2048 workgroups:
//   64 features:   one causal document .33 - .49 | .37 - .51 | .53 - .64 | .60 - .70     ragged, mean 100 - 800 | | .59 - .80 | .61 - .86
//                  not causal .41 - .58 | .62 - .73 | .90 - .96 | 1.06 - 1.18            documents of 512 .47 | .70 - .78 | | .91 - 1.06
//   128 features:  causal .38 - .53 | .51 - .84 | .72 - 1.06 | .91 - 1.2      not causal .50 - .78 | .87 - 1.10 | 1.3 | 1.5
// (4 / 4, 12 / 12, 16 / 4 and 32 / 8 heads, the rows that make up the count; 1 and 2 heads with documents of up to 65536 tokens alike: the
// length of a context alone does not decide.)  us at some of these, tiled / short: 32 / 8 heads of 128, 1024 tokens 34.7 / 23.9; 16 heads of
// 128, 8 documents of 512: 29.3 / 41.3; 12 heads of 64, 3001 tokens in documents of 17 - 400: 20.9 / 12.3; 1 head of 64, 65536 tokens: 1280 / 762.
// Up to 128 rows are a single workgroup per head and a chain of two key tiles in the tiled kernels: 8.0 / 5.0 us forward and 20 / 14
// backward (100 rows, 2 heads of 64), both less than the host takes to issue them; such calls stay where they were.
static inline bool mi_attn_fwd_is_short(const mi_attn_args* a) {
    if (a->flags & (MI_ATTN_QG1 | MI_ATTN_QG2 | MI_ATTN_TILED)) return false;
    if (a->flags & MI_ATTN_SHORT) return true;
    const int64_t rows = a->total_q > a->total_k ? a->total_q : a->total_k, blocks = mi_attn_short_blocks(a, a->n_q_heads), units = mi_compute_units();
    const int64_t per_unit = a->head_dim <= 64 ? (a->causal ? 8 : 6) : (a->causal ? 4 : 3);
    if (rows <= 128) return false;
    if (blocks <= per_unit * units) return true;
    // More blocks, of short documents and with two wavefronts each: two / tiled .42 - 1.01, mean .76 (32 heads of 64, 8192 tokens, documents of 20 - 380 47.1 / 64.2 us; 16 heads of
    // 128 43.9 / 50.3).  Not where k is rotated here: these blocks rotate a tile more often.
    const int64_t chain = (a->causal ? 1 : 2) * rows / (a->n_docs > 1 ? a->n_docs : 1);
    return mi_attn_short_pairs(a, false, blocks) && (a->rotary_cos == nullptr || a->position_ids_k == nullptr) &&
           (a->head_dim <= 64 ? chain <= (a->causal ? 600 : 400) : chain <= 250 && blocks <= 32 * units);
}

// The same for a backward pass, whose blocks of either kind (dQ: rows / 32 x query heads, dK / dV: rows / 32 x KV heads x head split)
// share a launch here as they do in the tiled kernels.  Short / tiled, over 510 calls of 1 - 32 heads drawn between 130 and 16384 tokens:
//   up to 64 features, where a compute unit holds three blocks of either kind, by dQ blocks:
//     up to 1500 .35 - .97          1500 - 2600 .71 - .99 (not causal 1.02 - 1.07, 8 documents of 256 1.26)
//     2600 - 4100: one document .93 - 1.13, ragged documents of 30 - 500 .78 - .94          4100 - 7000: 1.02 - 1.12, ragged .78 - .90
//   above, where one block fills it, by blocks of both kinds, causal, without | with groups of 4 query heads:
//     350 .63 - .88 | .60       500 .67 - .96 | .61       576 .77 - 1.0 | .65      640 .95 - 1.15 | .62 - .68     760 .97 - 1.15 | .79 - .84     1120 1.1 | .97
//     one causal document, whose chain the tiled kernels walk alone: 700 .89, 770 .74, 900 .86, 1060 1.11
// Of the 510 the rule takes 12 to the slower side, by 2 - 8 %.  us, tiled / short: 12 heads of 64, 3001 tokens in documents of 17 - 400:
// 35.9 / 31.3; 32 / 8 heads of 128, 512 tokens 57.4 / 35.5; 4 heads of 64, 1024 tokens 29.2 / 17.0.
// Longer chains above 64 features are a band of their own: there dQ blocks are better off two to a compute unit, in a launch in front of the
// dK / dV blocks (tiled / together / apart, us: 16 / 4 heads of 128, 1664 tokens 95 / 105 / 90; 32 / 8, 1316 tokens 137 / 134 / 124; 32 / 1,
// 3 documents of 312 64 / 64 / 59).
enum class ShortBwd { kNo, kTogether, kApart };
static inline ShortBwd mi_attn_bwd_short(const mi_attn_args* a, int hsplit) {
    if (a->flags & (MI_ATTN_QG1 | MI_ATTN_QG2 | MI_ATTN_TILED)) return ShortBwd::kNo;
    if (a->flags & MI_ATTN_SHORT) return ShortBwd::kTogether;
    const int64_t rows = a->total_q > a->total_k ? a->total_q : a->total_k, docs = a->n_docs > 1 ? a->n_docs : 1, units = mi_compute_units();
    if (rows <= 128) return ShortBwd::kNo;
    const int64_t row_blocks = (rows + kShortRows - 1) / kShortRows, dq = row_blocks * a->n_q_heads, both = dq + row_blocks * a->n_kv_heads * hsplit;
    const int64_t group = a->n_q_heads / a->n_kv_heads / hsplit;                                      // query heads of a dK / dV block
    const bool causal = a->causal != 0;
    const bool whole = a->total_q == a->total_k && rows % (256 * docs) == 0;                          // may be whole tiled blocks, all of them
    const bool chains = causal && (whole ? rows >= 1024 * docs * docs : rows >= 512 * docs);        // the chain of a document dominates
    if (a->head_dim <= 64) {
        int64_t per_unit_8;                                                                           // 8 x dQ blocks per compute unit
        if (!whole && docs > 1 && rows <= 512 * docs) per_unit_8 = 192;
        else if (causal && (!whole || chains)) per_unit_8 = 80 + 12 * (group - 1) < 96 ? 80 + 12 * (group - 1) : 96;
        else per_unit_8 = (causal ? 32 : 40) + 12 * (group - 1) < 64 ? (causal ? 32 : 40) + 12 * (group - 1) : 64;
        if (dq * 8 <= per_unit_8 * units) return ShortBwd::kTogether;
        // two wavefronts / tiled .68 - 1.00, mean .81: 32 heads of 64, documents of 20 - 380, 4096 tokens 68.5 / 101 us, 8192 144 / 181
        return mi_attn_short_pairs(a, true, both) && a->n_q_heads >= 16 && (causal ? 1 : 2) * rows <= 400 * docs ? ShortBwd::kTogether : ShortBwd::kNo;
    }
    const bool alone = chains && rows >= 1024 * docs * docs;                                         // few documents, long ones
    int64_t eighths = whole && docs > 1 && !chains ? 16 : 18 + 9 * (group - 1) / 2;                              // of a block of either kind per compute unit
    if (alone && eighths < 28) eighths = 28;
    if (both * 8 <= eighths * units) return ShortBwd::kTogether;
    if (causal && rows * group >= (group < 4 ? 1536 : 1024) * docs && (alone || group >= 4) && both <= (3 + group) * units) return ShortBwd::kApart;
    return ShortBwd::kNo;
}

// ---- forward: 32 queries of one head --------------------------------------------------------------------------------
// QROT: 0 = q as it is, 1 = rotate-half, 2 = interleaved rotary on the q load; KROT: k is rotated too, in its LDS tile (otherwise it
// arrives rotated, as training passes it)
template <int D, int QROT, bool KROT, int WAVES>
__global__ __launch_bounds__(64 * WAVES, D <= 64 ? 4 : 2) void attn_short_fwd_kernel(const AttnParams p) {
    constexpr int KS = D / 16, DT = D / 32;
    using Stages = ShortStages<D, WAVES>;
    using Tile = LdsTile<D>;
    constexpr int RB = Tile::RB;
    constexpr int kRed = kShortRed<D, WAVES>;
    __shared__ __attribute__((aligned(1024))) char smem[Stages::kSmem > kRed ? Stages::kSmem : kRed];
    __shared__ float m_lds[WAVES][32], l_lds[WAVES][32];
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nqb = (p.total_q + 31) / 32;
    int head, rank;
    head_and_rank(blockIdx.x, p.nq, head, rank);
    const int qb = nqb - 1 - rank, kvh = head / p.n_rep;
    const int tq = qb * 32 + l32, tl = min(tq, p.total_q - 1);

    elem8_t qf[KS];
    {
        const elem_t* qrow = p.q + (int64_t)tl * p.q_st + (int64_t)head * p.q_sh + 8 * g;
        uint4 raw[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) raw[ks] = ld128(qrow + 16 * ks);
        if constexpr (QROT != 0) {
            int64_t pos = p.pos_q[tl];
            pos = pos < 0 ? 0 : (pos >= p.table_rows ? p.table_rows - 1 : pos);
            if constexpr (QROT == 1) {
#pragma unroll
                for (int ks = 0; ks < KS / 2; ++ks)
                    rotate_pair(raw[ks], raw[ks + KS / 2], ld128(p.cos + pos * D + 16 * ks + 8 * g), ld128(p.sin + pos * D + 16 * ks + 8 * g), 1.0f);
            } else {
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
                    rotate_interleaved(raw[ks], ld128(p.cos32 + pos * (D / 2) + 8 * ks + 4 * g), ld128(p.sin32 + pos * (D / 2) + 8 * ks + 4 * g), 1.0f);
            }
            if (p.q_rot != nullptr && wave == 0 && tq < p.total_q) {
                elem_t* qo = p.q_rot + (int64_t)tq * p.q_st + (int64_t)head * p.q_sh + 8 * g;
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) st128(qo + 16 * ks, raw[ks]);
            }
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qf[ks] = __builtin_bit_cast(elem8_t, raw[ks]);
    }
    int klo, khi, wmin, wmax, kt0, n_tiles;
    short_key_range(p, tq, lane, klo, khi);
    short_tiles(klo, khi, wmin, wmax, kt0, n_tiles);

    f32x16_t o_acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o_acc[dt][r] = 0.f;
    float m_i = -INFINITY, l_i = 0.f;

    const Stages st{smem + wave * Stages::kBytes};
    const elem_t* kbase = p.k + (int64_t)kvh * p.k_sh;
    const elem_t* vbase = p.v + (int64_t)kvh * p.v_sh;
    DmaPlan<D, Stages::kLoads> k_plan, v_plan;
    k_plan.init(0, lane, p.k_st);
    v_plan.init(0, lane, p.v_st);
    auto issue_k = [&](int tile) { k_plan.issue(kbase, p.k_st, kt0 + 32 * tile, p.total_k - 1, st.first()); };
    auto issue_v = [&](int tile) { v_plan.issue(vbase, p.v_st, kt0 + 32 * tile, p.total_k - 1, st.second()); };
    const char *ks_ = st.first(), *vs_ = st.second();
    int h0, h1;
    Tile::tr_bases(lane, h0, h1);
    const int k_row = Tile::row_base(l32, g);
    if (wave < n_tiles) { issue_k(wave); issue_v(wave); }
    for (int tile = wave; tile < n_tiles; tile += WAVES) {
        const bool next = tile + WAVES < n_tiles;
        const int kt = kt0 + 32 * tile;
        wait_vmcnt<Stages::kLoads>();     // K has landed, V may still be in flight
        if constexpr (KROT) {
#pragma unroll
            for (int j = 0; j < D / 32; ++j) {
                const int row = (lane + 64 * j) / (D / 16), c = (lane + 64 * j) % (D / 16);
                char *at0 = st.first() + Tile::unit_offset(row, c), *at1 = st.first() + Tile::unit_offset(row, c + D / 16);
                uint4 lo = ld128(at0), hi = ld128(at1);
                int64_t pos = p.pos_k[min(kt + row, p.total_k - 1)];
                pos = pos < 0 ? 0 : (pos >= p.table_rows ? p.table_rows - 1 : pos);
                if constexpr (QROT == 1) {
                    rotate_pair(lo, hi, ld128(p.cos + pos * D + 8 * c), ld128(p.sin + pos * D + 8 * c), 1.0f);
                } else {
                    const float *cr = p.cos32 + pos * (D / 2) + 4 * c, *sr = p.sin32 + pos * (D / 2) + 4 * c;
                    rotate_interleaved(lo, ld128(cr), ld128(sr), 1.0f);
                    rotate_interleaved(hi, ld128(cr + D / 4), ld128(sr + D / 4), 1.0f);
                }
                st128(at0, lo);
                st128(at1, hi);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
        f32x16_t s_acc;
#pragma unroll
        for (int r = 0; r < 16; ++r) s_acc[r] = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) s_acc = mfma_32x32x16(*reinterpret_cast<const elem8_t*>(ks_ + (k_row ^ (ks << 5))), qf[ks], s_acc);
        Stages::reads_done();
        if (next) issue_k(tile + WAVES);
        // rows of the accumulator are keys kt + 8 a + 4 g + c, the column is this lane's query
        if (__any((kt < klo) || (kt + 32 > khi))) {
            const int rel0 = kt + 4 * g - klo;
            const unsigned len = (unsigned)(khi - klo);
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if ((unsigned)(rel0 + 8 * (r >> 2) + (r & 3)) >= len) s_acc[r] = -INFINITY;
        }
        float mx = s_acc[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s_acc[r]);
        const float m_new = fmaxf(m_i, pair_max(mx) * p.scale_log2);
        if (__any(m_new > m_i)) {
            const float alpha = m_new == -INFINITY ? 1.0f : fast_exp2(m_i - m_new);
            m_i = m_new;
            l_i *= alpha;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) o_acc[dt][r] *= alpha;
        }
        const float m_use = m_i == -INFINITY ? 0.f : m_i;
        elem8_t pf[2];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float e = fast_exp2(s_acc[r] * p.scale_log2 - m_use);
            l_i += e;
            pf[r >> 3][r & 7] = (elem_t)e;
        }
        if (next) wait_vmcnt<Stages::kLoads>(); else wait_vmcnt<0>();     // V has landed, the next K may be in flight
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
                o_acc[dt] = mfma_32x32x16(tr_pair(vs_ + (h0 ^ (dt << 6)) + 16 * m * RB, vs_ + (h1 ^ (dt << 6)) + 16 * m * RB), pf[m], o_acc[dt]);
        Stages::reads_done();
        if (next) issue_v(tile + WAVES);
    }
    // ---- merge
    l_i = pair_sum(l_i);
    if (g == 0) { m_lds[wave][l32] = m_i; l_lds[wave][l32] = l_i; }
    __syncthreads();
    float M = -INFINITY, L = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) M = fmaxf(M, m_lds[w][l32]);
#pragma unroll
    for (int w = 0; w < WAVES; ++w) L += m_lds[w][l32] == -INFINITY ? 0.f : l_lds[w][l32] * fast_exp2(m_lds[w][l32] - M);
    const float f = m_i == -INFINITY ? 0.f : fast_exp2(m_i - M);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o_acc[dt][r] *= f;
    float* red = reinterpret_cast<float*>(smem);
    short_store<D>(red, wave, lane, o_acc);
    __syncthreads();
    if (tq >= p.total_q) return;
    float x[4 / WAVES][DT][4];
    short_sums<D, WAVES>(red, wave, lane, x);
#pragma unroll
    for (int j = 0; j < 4 / WAVES; ++j)
        short_write<D>(p.o + (int64_t)tq * p.o_st + (int64_t)head * p.o_sh + 8 * (wave * (4 / WAVES) + j) + 4 * g, x[j], L > 0.f ? 1.0f / L : 0.f);
    if (wave == 0 && g == 0 && p.lse != nullptr)
        p.lse[(int64_t)head * p.total_q + tq] = L > 0.f ? (M + __log2f(L)) * 0.6931471805599453f : INFINITY;
}

// acc + the products of eight features of an O row and a dO row: delta = sum of them over the features, in the same order wherever
// these kernels form it
__device__ __forceinline__ float short_dot(const elem8_t& o, const elem8_t& d_o, float acc) {
    float a[8], b[8];
    Elem<elem_t>::unpack(__builtin_bit_cast(uint4, o), a);
    Elem<elem_t>::unpack(__builtin_bit_cast(uint4, d_o), b);
#pragma unroll
    for (int i = 0; i < 8; ++i) acc += a[i] * b[i];
    return acc;
}

// delta for the dK / dV blocks of long chains, in a launch in front: two lanes per (token, head) row, its sums in the order of the blocks that form
// their own, so that a gradient does not depend on who formed its delta.  (The tiled kernels' 16 lanes sum in another order.)
template <int D>
__global__ __launch_bounds__(256) void attn_bwd_delta_short_kernel(const AttnParams p) {
    const int64_t item = (int64_t)blockIdx.x * 256 + threadIdx.x, row = item >> 1;
    if (row >= (int64_t)p.total_q * p.nq) return;          // both lanes of a row
    const int64_t t = row / p.nq;
    const int h = (int)(row - t * p.nq), g = (int)(item & 1);
    const elem_t *o = p.o + t * p.o_st + (int64_t)h * p.o_sh + 8 * g, *d_o = p.d_o + t * p.o_st + (int64_t)h * p.o_sh + 8 * g;
    elem8_t a[D / 16], b[D / 16];
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
        a[ks] = *reinterpret_cast<const elem8_t*>(o + 16 * ks);
        b[ks] = *reinterpret_cast<const elem8_t*>(d_o + 16 * ks);
    }
    float delta = 0.f;
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) delta = short_dot(a[ks], b[ks], delta);
    delta = group_sum<2>(delta);
    if (g == 0) p.delta[(int64_t)h * p.total_q + t] = delta;
}

// ---- backward: dQ of 32 queries of one head ------------------------------------------------------------------
template <int D, int WAVES> constexpr int kShortDqSmem = ShortStages<D, WAVES>::kSmem < kShortRed<D, WAVES> ? kShortRed<D, WAVES> : ShortStages<D, WAVES>::kSmem;

template <int D, int WAVES, bool KEEP_DELTA>
__device__ __forceinline__ void short_dq_block(const AttnParams& p, char* smem, int block) {
    constexpr int KS = D / 16, DT = D / 32;
    using Stages = ShortStages<D, WAVES>;
    using Tile = LdsTile<D>;
    constexpr int RB = Tile::RB;
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nqb = (p.total_q + 31) / 32;
    int head, rank;
    head_and_rank(block, p.nq, head, rank);
    const int qb = nqb - 1 - rank, kvh = head / p.n_rep;
    const int tq = qb * 32 + l32, tl = min(tq, p.total_q - 1);

    elem8_t qf[KS], dof[KS];
    float delta = 0.f;
    {
        const elem_t* qr = p.q + (int64_t)tl * p.q_st + (int64_t)head * p.q_sh + 8 * g;
        const elem_t* dr = p.d_o + (int64_t)tl * p.o_st + (int64_t)head * p.o_sh + 8 * g;
        const elem_t* orow = p.o + (int64_t)tl * p.o_st + (int64_t)head * p.o_sh + 8 * g;
        uint4 o_raw[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            qf[ks] = __builtin_bit_cast(elem8_t, ld128(qr + 16 * ks));
            dof[ks] = __builtin_bit_cast(elem8_t, ld128(dr + 16 * ks));
            o_raw[ks] = ld128(orow + 16 * ks);
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) delta = short_dot(__builtin_bit_cast(elem8_t, o_raw[ks]), dof[ks], delta);
        delta = pair_sum(delta);
        if (KEEP_DELTA && wave == 0 && g == 0 && tq < p.total_q) p.delta[(int64_t)head * p.total_q + tq] = delta;
    }
    const float lse2 = p.lse[(int64_t)head * p.total_q + tl] * 1.4426950408889634f;
    int klo, khi, wmin, wmax, kt0, n_tiles;
    short_key_range(p, tq, lane, klo, khi);
    short_tiles(klo, khi, wmin, wmax, kt0, n_tiles);

    f32x16_t dq_acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) dq_acc[dt][r] = 0.f;
    const Stages st{smem + wave * Stages::kBytes};
    const elem_t* kbase = p.k + (int64_t)kvh * p.k_sh;
    const elem_t* vbase = p.v + (int64_t)kvh * p.v_sh;
    DmaPlan<D, Stages::kLoads> k_plan, v_plan;
    k_plan.init(0, lane, p.k_st);
    v_plan.init(0, lane, p.v_st);
    auto issue_k = [&](int tile) { k_plan.issue(kbase, p.k_st, kt0 + 32 * tile, p.total_k - 1, st.first()); };
    auto issue_v = [&](int tile) { v_plan.issue(vbase, p.v_st, kt0 + 32 * tile, p.total_k - 1, st.second()); };
    const char *ks_ = st.first(), *vs_ = st.second();
    int h0, h1;
    Tile::tr_bases(lane, h0, h1);
    const int a_row = Tile::row_base(l32, g);
    if (wave < n_tiles) { issue_v(wave); issue_k(wave); }
    for (int tile = wave; tile < n_tiles; tile += WAVES) {
        const bool next = tile + WAVES < n_tiles;
        const int kt = kt0 + 32 * tile;
        wait_vmcnt<0>();
        f32x16_t s_acc, dp_acc;
#pragma unroll
        for (int r = 0; r < 16; ++r) { s_acc[r] = 0.f; dp_acc[r] = 0.f; }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            s_acc = mfma_32x32x16(*reinterpret_cast<const elem8_t*>(ks_ + (a_row ^ (ks << 5))), qf[ks], s_acc);
            dp_acc = mfma_32x32x16(*reinterpret_cast<const elem8_t*>(vs_ + (a_row ^ (ks << 5))), dof[ks], dp_acc);
        }
        Stages::reads_done();
        if (next) issue_v(tile + WAVES);
        if (__any((kt < klo) || (kt + 32 > khi))) {
            const int rel0 = kt + 4 * g - klo;
            const unsigned len = (unsigned)(khi - klo);
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if ((unsigned)(rel0 + 8 * (r >> 2) + (r & 3)) >= len) s_acc[r] = -INFINITY;
        }
        elem8_t dsf[2];
#pragma unroll
        for (int r = 0; r < 16; ++r) dsf[r >> 3][r & 7] = (elem_t)(fast_exp2(s_acc[r] * p.scale_log2 - lse2) * (dp_acc[r] - delta));
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
                dq_acc[dt] = mfma_32x32x16(tr_pair(ks_ + (h0 ^ (dt << 6)) + 16 * m * RB, ks_ + (h1 ^ (dt << 6)) + 16 * m * RB), dsf[m], dq_acc[dt]);
        Stages::reads_done();
        if (next) issue_k(tile + WAVES);
    }
    __syncthreads();                      // every wavefront is done with its stages
    float* red = reinterpret_cast<float*>(smem);
    short_store<D>(red, wave, lane, dq_acc);
    __syncthreads();
    if (tq >= p.total_q) return;
    float x[4 / WAVES][DT][4];
    short_sums<D, WAVES>(red, wave, lane, x);
#pragma unroll
    for (int j = 0; j < 4 / WAVES; ++j) {
        const int a = wave * (4 / WAVES) + j;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int c = 0; c < 4; ++c) x[j][dt][c] *= p.scale;
        if constexpr (D == 64 || D == 128) {
            if (p.unrotate != 0) short_unrotate<D>(x[j], p, p.pos_q[tq], a, g);
        }
        short_write<D>(p.dq + (int64_t)tq * p.q_st + (int64_t)head * p.q_sh + 8 * a + 4 * g, x[j], 1.0f);
    }
}

// ---- backward: dK and dV of 32 keys of one KV head (of one share of its query heads: hsplit) ------------------------------
// The wavefronts take (query tile, query head) pairs in turn.  OWN_DELTA: they form delta themselves, from the fragments of the dO tile and of
// an O tile (up to 64 features) or of O rows in registers, which a compute unit's only workgroup has enough of; otherwise a launch in front has left it.
template <int D, int WAVES, bool OWN_DELTA> using ShortDkdvStages = ShortStages<D, WAVES, D <= 64 ? 1 : 2, OWN_DELTA && D <= 64 ? 3 : 2>;
template <int D, int WAVES, bool OWN_DELTA>
constexpr int kShortDkdvSmem = ShortDkdvStages<D, WAVES, OWN_DELTA>::kSmem < kShortRed<D, WAVES> ? kShortRed<D, WAVES>
                                                                                                          : ShortDkdvStages<D, WAVES, OWN_DELTA>::kSmem;

// stat_lds: 32 log-sum-exps, 32 deltas of each wavefront's tile
template <int D, int WAVES, bool OWN_DELTA>
__device__ __forceinline__ void short_dkdv_block(const AttnParams& p, char* smem, float (*stat_lds)[64], int block) {
    constexpr int KS = D / 16, DT = D / 32;
    constexpr int STAGES = D <= 64 ? 1 : 2;
    constexpr bool O_TILE = OWN_DELTA && D <= 64, O_ROWS = OWN_DELTA && D > 64;
    using Stages = ShortDkdvStages<D, WAVES, OWN_DELTA>;
    using Tile = LdsTile<D>;
    constexpr int RB = Tile::RB;
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int group, kb;
    head_and_rank(block, p.nkv * p.hsplit, group, kb);            // key blocks with the most queries come first
    const int kvh = group / p.hsplit, hs = group - kvh * p.hsplit, hpw = p.n_rep / p.hsplit;
    const int key = kb * 32 + l32, kl = min(key, p.total_k - 1);

    elem8_t kf[KS], vf[KS];
    {
        const elem_t* kr = p.k + (int64_t)kl * p.k_st + (int64_t)kvh * p.k_sh + 8 * g;
        const elem_t* vr = p.v + (int64_t)kl * p.v_st + (int64_t)kvh * p.v_sh + 8 * g;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            kf[ks] = __builtin_bit_cast(elem8_t, ld128(kr + 16 * ks));
            vf[ks] = __builtin_bit_cast(elem8_t, ld128(vr + 16 * ks));
        }
    }
    int qlo, qhi, wmin, wmax, qt0, n_tiles;
    short_query_range(p, key, lane, qlo, qhi);
    short_tiles(qlo, qhi, wmin, wmax, qt0, n_tiles);

    f32x16_t dk_acc[DT], dv_acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) { dk_acc[dt][r] = 0.f; dv_acc[dt][r] = 0.f; }
    const Stages st{smem + wave * Stages::kBytes};
    DmaPlan<D, Stages::kLoads> q_plan, do_plan;
    q_plan.init(0, lane, p.q_st);
    do_plan.init(0, lane, p.o_st);
    const int iters = n_tiles * hpw;
    const float* stat_base = OWN_DELTA || g == 0 ? p.lse : p.delta;
    const float stat_scale = OWN_DELTA || g == 0 ? 1.4426950408889634f : 1.0f;
    float stat = 0.f;
    elem8_t o_raw[O_ROWS ? KS : 1];
    auto issue = [&](int iter, int buf) {
        const int tile = iter / hpw, head = kvh * p.n_rep + hs * hpw + (iter - tile * hpw), qt = qt0 + 32 * tile;
        stat = stat_base[(int64_t)head * p.total_q + min(qt + l32, p.total_q - 1)];
        q_plan.issue(p.q + (int64_t)head * p.q_sh, p.q_st, qt, p.total_q - 1, st.first(buf));
        do_plan.issue(p.d_o + (int64_t)head * p.o_sh, p.o_st, qt, p.total_q - 1, st.second(buf));
        if constexpr (O_TILE) do_plan.issue(p.o + (int64_t)head * p.o_sh, p.o_st, qt, p.total_q - 1, st.third(buf));
    };
    auto load_o = [&](int iter) {
        const int tile = iter / hpw, head = kvh * p.n_rep + hs * hpw + (iter - tile * hpw);
        const elem_t* row = p.o + (int64_t)min(qt0 + 32 * tile + l32, p.total_q - 1) * p.o_st + (int64_t)head * p.o_sh + 8 * g;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) o_raw[ks] = *reinterpret_cast<const elem8_t*>(row + 16 * ks);
    };
    int h0, h1;
    Tile::tr_bases(lane, h0, h1);
    const int a_row = Tile::row_base(l32, g);
    if (wave < iters) {
        issue(wave, 0);
        if constexpr (O_ROWS) load_o(wave);
    }
    int buf = 0;
    for (int iter = wave; iter < iters; iter += WAVES) {
        const bool next = iter + WAVES < iters;
        if (!OWN_DELTA || g == 0) stat_lds[wave][lane] = stat * stat_scale;
        if constexpr (O_ROWS) {                           // waited for here, or the wait would take the next step's tiles along
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(o_raw[ks]));
        }
        const char *qs_ = st.first(buf), *ds_ = st.second(buf);
        if (STAGES == 2 && next) {
            issue(iter + WAVES, buf ^ 1);
            wait_vmcnt<2 * Stages::kLoads>();             // this step's tiles and rows have landed, the next one's tiles may be in flight
        } else {
            wait_vmcnt<0>();
        }
        if constexpr (OWN_DELTA) {
            float delta = 0.f;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const int at = a_row ^ (ks << 5);
                const elem8_t d_o = *reinterpret_cast<const elem8_t*>(ds_ + at);
                if constexpr (O_TILE) delta = short_dot(*reinterpret_cast<const elem8_t*>(st.third(buf) + at), d_o, delta);
                else delta = short_dot(o_raw[ks], d_o, delta);
            }
            delta = pair_sum(delta);
            if (g == 1) stat_lds[wave][lane] = delta;
            __builtin_amdgcn_sched_barrier(0);            // before the accumulators are live: 168 registers at 64 features
            if constexpr (O_ROWS) {
                if (next) load_o(iter + WAVES);
            }
        }
        const int qs = qt0 + 32 * (iter / hpw);
        f32x16_t s_acc, dp_acc;
#pragma unroll
        for (int r = 0; r < 16; ++r) { s_acc[r] = 0.f; dp_acc[r] = 0.f; }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            s_acc = mfma_32x32x16(*reinterpret_cast<const elem8_t*>(qs_ + (a_row ^ (ks << 5))), kf[ks], s_acc);
            dp_acc = mfma_32x32x16(*reinterpret_cast<const elem8_t*>(ds_ + (a_row ^ (ks << 5))), vf[ks], dp_acc);
        }
        // rows of the accumulators are queries qs + 8 a + 4 g + c, the column is this lane's key
        if (__any((qs < qlo) || (qs + 32 > qhi))) {
            const int rel0 = qs + 4 * g - qlo;
            const unsigned len = (unsigned)(qhi - qlo);
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if ((unsigned)(rel0 + 8 * (r >> 2) + (r & 3)) >= len) s_acc[r] = -INFINITY;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");     // stat_lds: one wavefront's LDS accesses complete in program order
        elem8_t pf[2], dsf[2];
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const f32x4_t l4 = *reinterpret_cast<const f32x4_t*>(&stat_lds[wave][8 * a + 4 * g]);
            const f32x4_t d4 = *reinterpret_cast<const f32x4_t*>(&stat_lds[wave][32 + 8 * a + 4 * g]);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int r = 4 * a + c;
                const float pv = fast_exp2(s_acc[r] * p.scale_log2 - l4[c]);
                pf[r >> 3][r & 7] = (elem_t)pv;
                dsf[r >> 3][r & 7] = (elem_t)(pv * (dp_acc[r] - d4[c]));
            }
        }
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                const int o0 = (h0 ^ (dt << 6)) + 16 * m * RB, o1 = (h1 ^ (dt << 6)) + 16 * m * RB;
                dv_acc[dt] = mfma_32x32x16(tr_pair(ds_ + o0, ds_ + o1), pf[m], dv_acc[dt]);
                dk_acc[dt] = mfma_32x32x16(tr_pair(qs_ + o0, qs_ + o1), dsf[m], dk_acc[dt]);
            }
        Stages::reads_done();
        if (STAGES == 2) buf ^= 1;
        else if (next) issue(iter + WAVES, 0);
    }
    __syncthreads();                      // every wavefront is done with its stages
    float* red = reinterpret_cast<float*>(smem);
    short_store<D>(red, wave, lane, dk_acc);
    __syncthreads();
    float dk[4 / WAVES][DT][4], dv[4 / WAVES][DT][4];
    short_sums<D, WAVES>(red, wave, lane, dk);
    __syncthreads();
    short_store<D>(red, wave, lane, dv_acc);
    __syncthreads();
    if (key >= p.total_k) return;
    short_sums<D, WAVES>(red, wave, lane, dv);
#pragma unroll
    for (int j = 0; j < 4 / WAVES; ++j) {
        const int a = wave * (4 / WAVES) + j;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int c = 0; c < 4; ++c) dk[j][dt][c] *= p.scale;
        if (p.hsplit > 1) {
            const int64_t row = (((int64_t)hs * p.total_k + key) * p.nkv + kvh) * D + 8 * a + 4 * g;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                *reinterpret_cast<f32x4_t*>(p.dk_part + row + 32 * dt) = f32x4_t{dk[j][dt][0], dk[j][dt][1], dk[j][dt][2], dk[j][dt][3]};
                *reinterpret_cast<f32x4_t*>(p.dv_part + row + 32 * dt) = f32x4_t{dv[j][dt][0], dv[j][dt][1], dv[j][dt][2], dv[j][dt][3]};
            }
            continue;
        }
        if constexpr (D == 64 || D == 128) {
            if (p.unrotate != 0) short_unrotate<D>(dk[j], p, p.pos_k[key], a, g);
        }
        short_write<D>(p.dk + (int64_t)key * p.dk_st + (int64_t)kvh * p.dk_sh + 8 * a + 4 * g, dk[j], 1.0f);
        short_write<D>(p.dv + (int64_t)key * p.dv_st + (int64_t)kvh * p.dv_sh + 8 * a + 4 * g, dv[j], 1.0f);
    }
}

// Both in one launch: dK / dV blocks, the longer ones, in the first n_dkdv workgroups, dQ blocks in the others.
template <int D, int WAVES, bool OWN_DELTA>
__global__ __launch_bounds__(64 * WAVES, D <= 64 ? 3 : 1) void attn_short_bwd_kernel(const AttnParams p, int n_dkdv) {
    constexpr int kDq = kShortDqSmem<D, WAVES>, kDkdv = kShortDkdvSmem<D, WAVES, OWN_DELTA>;
    __shared__ __attribute__((aligned(1024))) char smem[kDq > kDkdv ? kDq : kDkdv];
    __shared__ __attribute__((aligned(16))) float stat_lds[WAVES][64];
    if ((int)blockIdx.x < n_dkdv) short_dkdv_block<D, WAVES, OWN_DELTA>(p, smem, stat_lds, blockIdx.x);
    else short_dq_block<D, WAVES, false>(p, smem, blockIdx.x - n_dkdv);
}

// dQ blocks alone, two to a compute unit; they leave delta for dK / dV
template <int D>
__global__ __launch_bounds__(256, 2) void attn_short_dq_kernel(const AttnParams p) {
    __shared__ __attribute__((aligned(1024))) char smem[kShortDqSmem<D, 4>];
    short_dq_block<D, 4, true>(p, smem, blockIdx.x);
}

}  // namespace
