// Decode attention over a pre-allocated KV cache for gfx950: one query token per sequence, HBM-bound.
//
// Grid = batch x KV heads x key splits.  All query heads of a GQA group are processed by the same
// workgroup, so every cached K/V element is read from HBM exactly once.  Each wavefront streams its
// own 32-key chunks:
//     S^T[key][head]  = K * Q^T     v_mfma_f32_16x16x32_bf16, A = K rows loaded straight from global
//                                   memory in operand layout, B = Q^T (heads of the group, zero padded)
//     online softmax over keys      the lane's column is a head; 8 in-lane keys + 2 lane exchanges
//     O^T[d][head]   += V^T * P^T   A = V^T read from a transposed per-wavefront LDS copy of the chunk
// Partial (max, sum, O) per split go to a workspace and are merged by the last workgroup of the splits to arrive (with tickets) or by a
// second kernel (none of it with a single split).
// The wavefront whose keys include the new token appends the new K/V row in place (instead of the
// reference's torch.cat), rotated, and puts the same bits into its operands of that chunk; the query is rotated while the
// first chunk is on its way.  (A launch of its own for the append took 3 - 5 us: a third of a step at batch 1.)
#include "attn_common.h"

#include <limits.h>

typedef float f32x4v __attribute__((ext_vector_type(4)));

namespace {

constexpr int kChunk = 32;           // keys per wavefront and iteration
constexpr int kMaxSplits = 32;

struct DecodeParams {
    const elem_t* q; elem_t* kc; elem_t* vc; elem_t* o;
    const int32_t* ctx_len;
    const elem_t* k_new; const elem_t* v_new;
    const elem_t* cos; const elem_t* sin; const int64_t* pos; int table_rows;
    const float* cos32; const float* sin32;   // interleaved-pair rotary: fp32 tables [table_rows, D / 2]
    int batch, max_ctx, nq, nkv, n_rep, n_splits;
    int n_hc;      // chunks of up to 16 query heads per KV head (a workgroup serves one chunk)
    uint32_t splits_m, groups_m, hc_m;   // for divide(): by n_splits, nkv * n_hc and n_hc
    int64_t c_sb, c_st, c_sh;
    int64_t q_sb, kn_sb, vn_sb;   // element strides between sequences of q / k_new / v_new
    float scale_log2;
    float* ws_o;   // [batch][nq][n_splits][D]
    float* ws_ml;  // [batch][nq][n_splits][2]
    int32_t* tickets;   // nullable: one arrival count per (batch, KV head, head chunk), zero between launches
};

__device__ __forceinline__ f32x4v mfma_16x16x32(elem8_t a, elem8_t b, f32x4v c) {
#ifdef MI_ELEM_F16
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
#else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
#endif
}

// Rotate-half rotary of a query or of the new key.  float16: sums are rounded once, but for features 2 - 7 of every eight of a key's second half, which are
// rounded to float32 first.  That is what the compiler once made of `rotate_pair` in either place, and what caches hold; it is named so that it no longer
// depends on the code around it.
template <bool KEY> __device__ __forceinline__ void rotate_row(uint4& lo, uint4& hi, const uint4& c, const uint4& s) {
#ifdef MI_ELEM_F16
    float x0[8], x1[8], cs[8], sn[8];
    Elem<elem_t>::unpack(lo, x0);
    Elem<elem_t>::unpack(hi, x1);
    Elem<elem_t>::unpack(c, cs);
    Elem<elem_t>::unpack(s, sn);
    uint32_t l[4], h[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int a = 2 * i, b = a + 1;
        l[i] = fma_pair_f16(x0[a], cs[a], -(x1[a] * sn[a]), x0[b], cs[b], -(x1[b] * sn[b]));
        h[i] = KEY && i > 0 ? pack_elem2(sum_f32(x1[a], cs[a], x0[a] * sn[a]), sum_f32(x1[b], cs[b], x0[b] * sn[b]))
                            : fma_pair_f16(x1[a], cs[a], x0[a] * sn[a], x1[b], cs[b], x0[b] * sn[b]);
    }
    lo = make_uint4(l[0], l[1], l[2], l[3]);
    hi = make_uint4(h[0], h[1], h[2], h[3]);
#else
    rotate_pair(lo, hi, c, s, 1.0f);
#endif
}

// ---- merge of the splits ------------------------------------------------------------------------------
// SHARED: the partial results pass between workgroups of one launch, past the L2s (those of the XCDs are not coherent; writing back and
// invalidating them, as a release and an acquire do, took 2 - 10 us of a launch of 104 - 256 workgroups).
template <bool SHARED> __device__ __forceinline__ float2 load_partial(const float* at) {
    if constexpr (!SHARED) return *reinterpret_cast<const float2*>(at);
    const uint64_t x = __hip_atomic_load(reinterpret_cast<const uint64_t*>(at), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return make_float2(__uint_as_float((uint32_t)x), __uint_as_float((uint32_t)(x >> 32)));
}
template <bool SHARED> __device__ __forceinline__ void store_partial(float* at, float x) {
    if constexpr (SHARED) __hip_atomic_store(at, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else *at = x;
}

// Features d and d + 1 of row bh = (batch, head), in steps of eight splits, the partial results of two steps requested before the first is
// used: 16 splits are one latency.
template <int D, bool SHARED>
__device__ __forceinline__ void merge_splits(const DecodeParams& p, int64_t bh, int d) {
    constexpr int kStep = 8, kSteps = 2;
    const float* ml = p.ws_ml + bh * p.n_splits * 2;
    const float* wo = p.ws_o + bh * p.n_splits * D + d;
    float M = -INFINITY, L = 0.f, O0 = 0.f, O1 = 0.f;
    for (int s0 = 0; s0 < p.n_splits; s0 += kSteps * kStep) {
        float2 mls[kSteps][kStep], os[kSteps][kStep];
#pragma unroll
        for (int h = 0; h < kSteps; ++h) {
            if (s0 + h * kStep >= p.n_splits) break;
#pragma unroll
            for (int i = 0; i < kStep; ++i) {              // past the last split: its values again, with no weight below
                const int s = min(s0 + h * kStep + i, p.n_splits - 1);
                mls[h][i] = load_partial<SHARED>(ml + 2 * s);
                os[h][i] = load_partial<SHARED>(wo + (int64_t)s * D);
            }
        }
#pragma unroll
        for (int h = 0; h < kSteps; ++h) {
            if (s0 + h * kStep >= p.n_splits) break;
            float m = M;
#pragma unroll
            for (int i = 0; i < kStep; ++i) m = fmaxf(m, mls[h][i].x);
            const float a = M == -INFINITY ? 0.f : fast_exp2(M - m);
            L *= a; O0 *= a; O1 *= a;
            M = m;
#pragma unroll
            for (int i = 0; i < kStep; ++i) {
                const float f = s0 + h * kStep + i >= p.n_splits || mls[h][i].x == -INFINITY ? 0.f : fast_exp2(mls[h][i].x - M);
                L += f * mls[h][i].y;
                O0 += f * os[h][i].x;
                O1 += f * os[h][i].y;
            }
        }
    }
    *reinterpret_cast<uint32_t*>(p.o + bh * D + d) = pack_elem2(L > 0.f ? O0 / L : 0.f, L > 0.f ? O1 / L : 0.f);
}

// ---- split kernel ----------------------------------------------------------------------------------
// NWV wavefronts (4 or 8) share the keys of one (batch, KV head, split); with a single split the merged result
// is the attention output and goes straight to `o`, otherwise the partial goes to the workspace.
// ROT: 0 = q as it is, 1 = rotate-half rotary on the q load, 2 = interleaved-pair rotary on the q load.
// BY_LENGTH: sequences are handed out by their lengths (order_by_length).  NEW_IN_LDS: the new row waits in LDS for its chunk (two_per_unit).
template <int D, int ROT, int NWV, bool BY_LENGTH, bool NEW_IN_LDS>
__global__ __launch_bounds__(64 * NWV, 2) void decode_split_kernel(const DecodeParams args) {
    constexpr int kThreads = 64 * NWV;
    constexpr int KS = D / 32;          // contraction steps of Q K^T (32 features each)
    constexpr int DT = D / 16;          // 16-row tiles of O^T
    constexpr int VSTR = 2 * D + 32;    // bytes per key row of the staged V chunk: transpose reads of 8 rows x 32 bytes hit 256 distinct bytes
    constexpr int V_ITEMS = 8 * (D / 8);  // (key quad, feature group) items of a 32-key chunk
    constexpr int V_PER_LANE = (V_ITEMS + 63) / 64;   // head_dim 32 / 96: the last round is partly empty

    __shared__ __attribute__((aligned(16))) char v_lds[NWV][kChunk * VSTR];
    __shared__ float wm_lds[NWV][16];
    __shared__ float wl_lds[NWV][16];
    __shared__ float wo_lds[NWV][16][D + 1];
    __shared__ __attribute__((aligned(16))) elem_t new_lds[2][NEW_IN_LDS ? D : 8];
    __shared__ int last_lds;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l16 = lane & 15, G = lane >> 4;

    // All arguments at once: read where they are used they are four trips of the scalar cache, one after the other, in front of the first load.
    DecodeParams p = args;
    arrived(p.q, p.kc, p.vc, p.o, p.ctx_len, p.k_new, p.v_new, p.max_ctx, p.nq, p.nkv, p.n_rep, p.n_splits, p.n_hc, p.splits_m, p.groups_m, p.hc_m);
    arrived(p.c_sb, p.c_st, p.c_sh, p.q_sb, p.kn_sb, p.vn_sb, p.scale_log2, p.ws_o, p.ws_ml, p.tickets);
    if constexpr (ROT == 1) arrived(p.cos, p.sin, p.pos, p.table_rows);
    if constexpr (ROT == 2) arrived(p.cos32, p.sin32, p.pos, p.table_rows);

    const int split = blockIdx.y;
    int b = divide(blockIdx.x, p.nkv * p.n_hc, p.groups_m);
    const int kv_hc = blockIdx.x - b * p.nkv * p.n_hc;
    const int kvh = divide(kv_hc, p.n_hc, p.hc_m), hc = kv_hc - kvh * p.n_hc;
    // this workgroup's query heads: head0 .. head0 + n_heads of the group (groups of more than 16 heads take
    // several workgroups, each reading the group's K / V once)
    const int head0 = kvh * p.n_rep + 16 * hc;
    const int n_heads = min(16, p.n_rep - 16 * hc);

    int ctx;
    int64_t pos = 0;                    // requested with ctx: the rows of the rotary tables need not wait for anything else
    if constexpr (!BY_LENGTH) {
        ctx = p.ctx_len[b];
        if constexpr (ROT != 0) pos = p.pos[b];
    } else {                            // lane i: sequence i; of different lengths the b-th shortest, in the last split the b-th longest
        const int n = args.batch, i = min(lane, n - 1), len = p.ctx_len[i];
        int64_t at = 0;
        if constexpr (ROT != 0) at = p.pos[i];
        if (__ballot(len != __builtin_amdgcn_readfirstlane(len)) != 0) {
            const int key = lane < n ? min(max(len, 0), p.max_ctx) * 64 + lane : INT_MAX;
            int rank = 0;
            for (int j = 0; j < n; j += 8)
#pragma unroll
                for (int u = 0; u < 8; ++u) rank += __builtin_amdgcn_readlane(key, j + u) < key;
            b = __builtin_ctzll(__ballot(lane < n && rank == (split == p.n_splits - 1 ? n - 1 - b : b)));
        }
        ctx = __builtin_amdgcn_readlane(len, b);
        if constexpr (ROT != 0)
            pos = (int64_t)((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(at >> 32), b) << 32 | (uint32_t)__builtin_amdgcn_readlane((int)at, b));
    }
    if constexpr (ROT != 0) pos = pos < 0 ? 0 : (pos >= p.table_rows ? p.table_rows - 1 : pos);
    const bool append = p.k_new != nullptr && ctx >= 1 && ctx <= p.max_ctx;
    ctx = ctx < 0 ? 0 : (ctx > p.max_ctx ? p.max_ctx : ctx);
    // keys of this split: [s0, s1), split length rounded up to whole workgroup iterations
    int per = divide(ctx + p.n_splits - 1, p.n_splits, p.splits_m);
    per = (per + NWV * kChunk - 1) / (NWV * kChunk) * (NWV * kChunk);
    const int s0 = split * per;
    const int s1 = min(ctx, s0 + per);
    const int n_iter = s1 > s0 ? (s1 - s0 + NWV * kChunk - 1) / (NWV * kChunk) : 0;

    // The last key of this split is the new token: the wavefront whose chunk (iteration it_new) holds it writes it to the cache and
    // replaces that key's operands, whose loads do not wait for the store and may bring what the row held before.  (Groups of more than 16 heads: each of
    // their workgroups does, with the same bytes, since each reads the row.)
    const int c_new = (ctx - 1 - s0) / kChunk;
    const int it_new = append && ctx - 1 >= s0 && ctx - 1 < s1 && c_new % NWV == wave ? c_new / NWV : -1;   // wave-uniform

    // A small call is a chain of trips to memory.  Whatever depends on nothing but ctx and pos is requested before the first of it is used, in the order of
    // use: q, the new row, rows of the rotary tables, the first chunk.  (With the arguments in one trip too, us in a graph, before / after: batch 1, 32 / 8
    // heads of 128, 1500 keys 7.9 / 7.3, 200 keys 6.7 / 5.9; batch 3, 16 / 4 of 64, 224 keys 5.1 / 4.3; batch 32, 32 / 8 of 128, 4096 keys 80.6 / 79.7.)
    // Q^T fragments: column = head slot l16 (valid when < n_rep), contraction = features 32*ks + 8*G + i; the new K row alike, in every column
    uint4 raw[KS], kn[KS] = {}, vn[V_PER_LANE] = {};
    {
        const int hs = l16 < n_heads ? l16 : 0;
        const elem_t* qr = p.q + (int64_t)b * p.q_sb + (int64_t)(head0 + hs) * D + 8 * G;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) raw[ks] = *reinterpret_cast<const uint4*>(qr + 32 * ks);
    }
    if (it_new >= 0) {
        const elem_t* kr = p.k_new + (int64_t)b * p.kn_sb + (int64_t)kvh * D + 8 * G;
        const elem_t* vr = p.v_new + (int64_t)b * p.vn_sb + (int64_t)kvh * D;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) kn[ks] = ld128(kr + 32 * ks);
#pragma unroll
        for (int j = 0; j < V_PER_LANE; ++j) vn[j] = ld128(vr + 8 * ((lane + 64 * j) % (D / 8)));
    }
    uint4 cv[KS / 2 + 1], sv[KS / 2 + 1];              // rotate-half: features 32 ks + 8 G .. + 8 of the first half
    uint4 ci[KS], si[KS];                              // interleaved: pairs 16 ks + 4 G .. + 4
    if constexpr (ROT == 1) {
#pragma unroll
        for (int ks = 0; ks < KS / 2; ++ks) {
            cv[ks] = ld128(p.cos + pos * D + 32 * ks + 8 * G);
            sv[ks] = ld128(p.sin + pos * D + 32 * ks + 8 * G);
        }
    } else if constexpr (ROT == 2) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            ci[ks] = ld128(p.cos32 + pos * (D / 2) + 16 * ks + 4 * G);
            si[ks] = ld128(p.sin32 + pos * (D / 2) + 16 * ks + 4 * G);
        }
    }

    f32x4v o_acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o_acc[dt] = f32x4v{0.f, 0.f, 0.f, 0.f};
    float m_i = -INFINITY, l_i = 0.f;

    const elem_t* kbase = p.kc + (int64_t)b * p.c_sb + (int64_t)kvh * p.c_sh;
    const elem_t* vbase = p.vc + (int64_t)b * p.c_sb + (int64_t)kvh * p.c_sh;
    char* vt = v_lds[wave];
    // transpose-read base of this lane: keys 4G + (l16 >> 2), features 4 * (l16 & 3) (+ 16 per feature tile, + 16 keys for the second half)
    const char* vt_lane = vt + (4 * G + (l16 >> 2)) * VSTR + 8 * (l16 & 3);

    // K fragments and V rows of a chunk; two sets so that the loads of chunk i+1 are in flight while
    // chunk i is being processed
    struct ChunkRegs {
        elem8_t kf[2][KS];
        uint4 vraw[V_PER_LANE][4];
    };
    // (a wavefront without keys asks for the last row or, of an empty cache, the first)
    auto request = [&](ChunkRegs& c, int it) {
        const int key0 = s0 + (NWV * it + wave) * kChunk, last = max(s1 - 1, 0);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int tok = min(key0 + 16 * t + l16, last);
            const elem_t* kr = kbase + (int64_t)tok * p.c_st + 8 * G;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) c.kf[t][ks] = __builtin_bit_cast(elem8_t, ldg_nt(reinterpret_cast<const uint4*>(kr + 32 * ks)));
        }
#pragma unroll
        for (int j = 0; j < V_PER_LANE; ++j) {
            const int item = lane + 64 * j;
            if (V_ITEMS % 64 != 0 && item >= V_ITEMS) break;
            const int quad = item / (D / 8), dg = item % (D / 8);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int tok = min(key0 + 4 * quad + r, last);
                c.vraw[j][r] = ldg_nt(reinterpret_cast<const uint4*>(vbase + (int64_t)tok * p.c_st + 8 * dg));
            }
        }
    };
    elem8_t qf[KS];
    // the new row in place of what its key (and keys past it, which read the same row) brought
    auto put_new = [&](ChunkRegs& c, int it) {
        const int key0 = s0 + (NWV * it + wave) * kChunk, last = s1 - 1;
        if constexpr (NEW_IN_LDS) {
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) kn[ks] = *reinterpret_cast<const uint4*>(new_lds[0] + 32 * ks + 8 * G);
#pragma unroll
            for (int j = 0; j < V_PER_LANE; ++j) vn[j] = *reinterpret_cast<const uint4*>(new_lds[1] + 8 * ((lane + 64 * j) % (D / 8)));
        }
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                if (key0 + 16 * t + l16 >= last) c.kf[t][ks] = __builtin_bit_cast(elem8_t, kn[ks]);
#pragma unroll
        for (int j = 0; j < V_PER_LANE; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (key0 + 4 * ((lane + 64 * j) / (D / 8)) + r >= last) c.vraw[j][r] = vn[j];
    };
    auto load_chunk = [&](ChunkRegs& c, int it) {
        if (s0 + (NWV * it + wave) * kChunk < s1) request(c, it);
    };
    auto process_chunk = [&](ChunkRegs& c, int it) {
        const int key0 = s0 + (NWV * it + wave) * kChunk;
        const bool active = key0 < s1;          // wave-uniform
        if (it == it_new) put_new(c, it);
        // Each wavefront owns its LDS chunk; the LDS pipeline executes one wavefront's accesses in program
        // order, so wavefront-scope fences (compiler ordering only) are enough and the wavefronts of a
        // workgroup never wait for each other inside the loop.
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        elem8_t pf;
        float alpha = 1.f;
        if (active) {
            f32x4v s_acc[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                s_acc[t] = f32x4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) s_acc[t] = mfma_16x16x32(c.kf[t][ks], qf[ks], s_acc[t]);
            }
            // rows: keys key0 + 16*t + 4*G + r; column: head slot l16
            float mx = -INFINITY;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (key0 + 16 * t + 4 * G + r >= s1) s_acc[t][r] = -INFINITY;
                    mx = fmaxf(mx, s_acc[t][r]);
                }
            mx = quad_max(mx);
            const float m_new = fmaxf(m_i, mx * p.scale_log2);   // finite: the chunk holds >= 1 valid key
            alpha = fast_exp2(m_i - m_new);
            m_i = m_new;
            float rs = 0.f;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float e = fast_exp2(s_acc[t][r] * p.scale_log2 - m_new);
                    rs += e;
                    pf[4 * t + r] = (elem_t)e;   // slot (G, i): key 16*(i/4) + 4*G + (i%4)
                }
            l_i = l_i * alpha + rs;
            // key-major copy of the V chunk (rows as loaded); the PV operand is read back transposed
#pragma unroll
            for (int j = 0; j < V_PER_LANE; ++j) {
                const int item = lane + 64 * j;
                if (V_ITEMS % 64 != 0 && item >= V_ITEMS) break;
                const int quad = item / (D / 8), dg = item % (D / 8);
#pragma unroll
                for (int r = 0; r < 4; ++r) st128(vt + (4 * quad + r) * VSTR + 16 * dg, c.vraw[j][r]);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (active) {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                // slots 0-3: keys 4G..4G+3, slots 4-7: keys 16+4G..16+4G+3 (the order of pf)
                const elem8_t a = tr_pair(vt_lane + 32 * dt, vt_lane + 16 * VSTR + 32 * dt);
                o_acc[dt] = o_acc[dt] * alpha;
                o_acc[dt] = mfma_16x16x32(a, pf, o_acc[dt]);
            }
        }
    };

    ChunkRegs ra, rb;
    __builtin_amdgcn_sched_barrier(0);                 // q, the new row and the tables first: their arrival is waited for alone
    request(ra, 0);                                    // without a branch, behind which q's arrival would be waited for as if this had not been sent
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (ROT == 1) {
#pragma unroll
        for (int ks = 0; ks < KS / 2; ++ks) {
            rotate_row<false>(raw[ks], raw[ks + KS / 2], cv[ks], sv[ks]);
            if (it_new >= 0) rotate_row<true>(kn[ks], kn[ks + KS / 2], cv[ks], sv[ks]);
        }
    } else if constexpr (ROT == 2) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            rotate_interleaved(raw[ks], ci[ks], si[ks], 1.0f);
            if (it_new >= 0) rotate_interleaved(kn[ks], ci[ks], si[ks], 1.0f);
        }
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        if (l16 >= n_heads) raw[ks] = make_uint4(0, 0, 0, 0);
        qf[ks] = __builtin_bit_cast(elem8_t, raw[ks]);
    }
    if (it_new >= 0) {
        const int64_t dst = (int64_t)b * p.c_sb + (int64_t)(ctx - 1) * p.c_st + (int64_t)kvh * p.c_sh;
        if (l16 == 0) {
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) st128(p.kc + dst + 32 * ks + 8 * G, kn[ks]);
        }
        if (lane < D / 8) st128(p.vc + dst + 8 * lane, vn[0]);
        if constexpr (NEW_IN_LDS) {                        // read back by the same wavefront
            if (l16 == 0) {
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) *reinterpret_cast<uint4*>(new_lds[0] + 32 * ks + 8 * G) = kn[ks];
            }
            if (lane < D / 8) *reinterpret_cast<uint4*>(new_lds[1] + 8 * lane) = vn[0];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        }
    }
    for (int it = 0; it < n_iter; it += 2) {
        if (it + 1 < n_iter) load_chunk(rb, it + 1);
        process_chunk(ra, it);
        if (it + 1 < n_iter) {
            if (it + 2 < n_iter) load_chunk(ra, it + 2);
            process_chunk(rb, it + 1);
        }
    }

    // ---- merge the four wavefronts, emit the split partial -----------------------------------------
    l_i = quad_sum(l_i);
    if (G == 0) { wm_lds[wave][l16] = m_i; wl_lds[wave][l16] = l_i; }
    if (l16 < n_heads) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int r = 0; r < 4; ++r) wo_lds[wave][l16][16 * dt + 4 * G + r] = o_acc[dt][r];
    }
    __syncthreads();
    for (int idx = tid; idx < n_heads * D; idx += kThreads) {
        const int hs = idx / D, d = idx % D;
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < NWV; ++w) M = fmaxf(M, wm_lds[w][hs]);
        float L = 0.f, O = 0.f;
#pragma unroll
        for (int w = 0; w < NWV; ++w) {
            const float wm = wm_lds[w][hs];
            const float f = wm == -INFINITY ? 0.f : fast_exp2(wm - M);
            L += f * wl_lds[w][hs];
            O += f * wo_lds[w][hs][d];
        }
        const int64_t bh = (int64_t)b * p.nq + head0 + hs;
        if (p.n_splits == 1) {
            p.o[bh * D + d] = (elem_t)(L > 0.f ? O / L : 0.f);
        } else {
            const int64_t slot = bh * p.n_splits + split;
            if (p.tickets != nullptr) {
                store_partial<true>(p.ws_o + slot * D + d, O);
                if (d == 0) { store_partial<true>(p.ws_ml + slot * 2, M); store_partial<true>(p.ws_ml + slot * 2 + 1, L); }
            } else {
                store_partial<false>(p.ws_o + slot * D + d, O);
                if (d == 0) { store_partial<false>(p.ws_ml + slot * 2, M); store_partial<false>(p.ws_ml + slot * 2 + 1, L); }
            }
        }
    }
    // With tickets the last workgroup of a (batch, KV head) to get here merges its splits; nobody waits for anybody.  The partial results are
    // stored past the L2 and every wavefront has waited for its own before the barrier, so the count that thread 0 raises behind it
    // comes after them in memory, and the loads of the workgroup that reads the highest count come after all.
    if (p.n_splits == 1 || p.tickets == nullptr) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
        int32_t* ticket = p.tickets + b * p.nkv * p.n_hc + kv_hc;
        const int arrived = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last_lds = arrived == p.n_splits - 1;
        if (arrived == p.n_splits - 1) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);     // for the next launch
    }
    __syncthreads();
    if (last_lds == 0) return;
    for (int idx = tid; idx < n_heads * (D / 2); idx += kThreads)
        merge_splits<D, true>(p, (int64_t)b * p.nq + head0 + idx / (D / 2), 2 * (idx % (D / 2)));
}

// Where the caller has no tickets: one thread per (batch, head, two features).  (With the append's launch gone as well, batch 1 over a cache of
// 1,024: 21.5 -> 11.2 us for a call; batch 32: 83.8 -> 81.6.)
template <int D>
__global__ __launch_bounds__(64) void decode_merge_kernel(const DecodeParams p) {
    const int64_t bh = (int64_t)blockIdx.x * (128 / D) + (2 * threadIdx.x) / D;
    const int d = (2 * threadIdx.x) % D;
    if (2 * threadIdx.x >= (128 / D) * D || bh >= (int64_t)p.batch * p.nq) return;
    merge_splits<D, false>(p, bh, d);
}

// Whether the last workgroup merges, given tickets.  On the device that is no gain: its one workgroup per (batch, KV head) loads past the caches what
// the merge launch spreads over more of them, with a thread for every two features of its heads and up to 16 splits 0 - 1 us more than that
// launch, beyond 2 - 9.  But a call of so few bytes is over before the host has issued two launches: batch 1, 32 / 8 heads of 128, a cache of 1,564, one call
// after the other 9.1 -> 7.6 us from C, 10.9 -> 8.8 from Python.
bool merges_in_launch(const DecodeParams& p, int head_dim) {
    const int heads = p.n_rep < 16 ? p.n_rep : 16;
    return p.n_splits > 1 && p.n_splits <= 16 && heads * head_dim <= 512 &&
           (int64_t)p.batch * p.nkv * p.max_ctx * head_dim * 4 <= (int64_t)32 << 20;
}

// 8-wavefront workgroups (one per compute unit) once there is a (batch, KV head) pair for most of the 256
// compute units, or when the whole cache is one 32-key chunk per wavefront or less: then one split does and the merge
// kernel is not launched; otherwise 4-wavefront workgroups and enough splits for about one workgroup per compute unit.
// One split / split and merge, microseconds, batch 1 with 32 query heads on 8, d 128: 6.1 / 6.8 with a cache of 256 tokens and
// 8.7 / 6.8 with 512; batch 8: 6.2 / 7.0 and 10.3 / 7.3; batch 3, 16 heads on 4, d 64: 4.4 / 5.5 and 5.6 / 5.5.
bool wide_blocks(int batch, int nkv, int max_ctx) { return (int64_t)batch * nkv >= 192 || max_ctx <= 8 * kChunk; }

int choose_splits(int batch, int nkv, int max_ctx) {
    const int64_t pairs = (int64_t)batch * nkv;
    if (wide_blocks(batch, nkv, max_ctx)) return 1;
    // one workgroup per compute unit: measured best or within a few percent of it for batch 1 - 16 at contexts
    // of 1k - 16k (two per compute unit, the earlier choice, cost 5 - 10 % in merge work at batch 4 - 16)
    int64_t s = (256 + pairs - 1) / pairs;
    const int64_t by_len = ((int64_t)max_ctx + 4 * kChunk - 1) / (4 * kChunk);
    if (s > by_len) s = by_len;
    if (s > kMaxSplits) s = kMaxSplits;
    if (s < 1) s = 1;
    return (int)s;
}

// Workgroups go to the compute units in the order of the grid: split 0 of every (sequence, KV head), then split 1 and so on.  Where there are more of them
// than compute units, the last, which are of the last split, join the first.  Splits are rounded up to whole iterations, so the last is the shortest, and
// sequences of one length gain from that order; of different lengths, long ones met by chance, and such a call lost more than it had gained.  So where
// workgroups share a compute unit, splits take the sequences from the shortest to the longest and the last split from the longest on: the units that get
// two of them get short ones.  us in a graph, bf16, splits of a sequence side by side / split by split / by length:
//   17 sequences of 2979 - 5956 keys, 32 / 8 heads of 128, 69.2 / 85.1 / 66.7     18 of 5977 - 11953 154 / 175 / 128     9 of 2979 - 5956 46.9 / 48.6 / 35.0
//   10 of up to 12472, 8 / 8 of 64, 33.8 / 39.8 / 33.1                            36 of up to 13740, 16 / 4 of 128, 171 / 189 / 119
//   17 of 4000, all of one length, 32 / 8 of 128, 76.9 / 75.8 / 75.6
// A workgroup finds its sequence among the lengths of all, one per lane, which is 0.3 us; with fewer than 512 keys a split there is no more than that
// to gain (344 keys: 12.7 split by split, 13.2 by length; 627: 15.4 / 13.3).  More than 64 sequences, with one or two KV heads, keep their order.
bool order_by_length(const DecodeParams& p) {
    const int64_t blocks = (int64_t)p.batch * p.nkv * p.n_hc * p.n_splits;
    return p.n_splits > 1 && p.batch > 1 && p.batch <= 64 && p.max_ctx >= 512 * p.n_splits && p.max_ctx < (1 << 24) && blocks > mi_compute_units();
}

// Whether 8-wavefront workgroups of 64 features, of which there are more than compute units, share these.  Two fit by LDS, but by registers only where the new row
// (K rotated, V) waits for its chunk in LDS instead: 119 registers, else 138.  One more trip through LDS is 0.1 - 0.2 us.  Long sequences are better off
// alone, the next one starting where the shortest has ended.  us in a graph, bf16, alone / shared:
//   57 sequences of 100 keys, 8 / 8 heads 7.3 / 6.7       30 of 800, 32 / 32 38.9 / 33.6       40 of 1200, 16 / 16 42.4 / 37.1
//   64 of 851 - 1700, 32 / 32 111.2 / 104.9               20 of 601 - 1200, 16 / 16 21.4 / 22.5   40 of 2500, 16 / 16 77.4 / 72.4
//   20 of up to 2500, 16 / 16 29.2 / 34.8                  57 of up to 4000, 8 / 8 62.5 / 66.4
template <int D> bool two_per_unit(const DecodeParams& p) {
    return D == 64 && (int64_t)p.batch * p.nkv * p.n_hc * p.n_splits > mi_compute_units() && p.max_ctx <= 2048;
}

// rot: 0 = none, 1 = rotate-half, 2 = interleaved pairs
template <int D, int NWV, bool BY_LENGTH, bool NEW_IN_LDS = false> int launch_split(const DecodeParams& p, int rot, hipStream_t st) {
    const dim3 grid((unsigned)p.batch * p.nkv * p.n_hc, p.n_splits), block(64 * NWV);
    if (rot == 2) decode_split_kernel<D, 2, NWV, BY_LENGTH, NEW_IN_LDS><<<grid, block, 0, st>>>(p);
    else if (rot == 1) {
        // rotate-half pairs feature i with i + D / 2: the same lane holds both only when D / 32 is even
        if constexpr (D == 64 || D == 128) decode_split_kernel<D, 1, NWV, BY_LENGTH, NEW_IN_LDS><<<grid, block, 0, st>>>(p);
        else return mi_fail(MI_E_SHAPE, "attn_decode: fused rotate-half rotary needs head_dim 64 or 128");
    } else decode_split_kernel<D, 0, NWV, BY_LENGTH, NEW_IN_LDS><<<grid, block, 0, st>>>(p);
    return mi_check_launch("decode_split");
}

template <int D> int launch_decode(const DecodeParams& p, int rot, hipStream_t st) {
    const bool wide = wide_blocks(p.batch, p.nkv * p.n_hc, p.max_ctx);
    const int rc = wide ? (two_per_unit<D>(p) ? launch_split<D, 8, false, D == 64>(p, rot, st) : launch_split<D, 8, false>(p, rot, st))
                        : (order_by_length(p) ? launch_split<D, 4, true>(p, rot, st) : launch_split<D, 4, false>(p, rot, st));
    if (rc != MI_OK || p.n_splits == 1 || p.tickets != nullptr) return rc;
    constexpr int kRows = 128 / D;
    const int64_t n = (int64_t)p.batch * p.nq;
    decode_merge_kernel<D><<<dim3((unsigned)((n + kRows - 1) / kRows)), dim3(64), 0, st>>>(p);
    return mi_check_launch("decode_merge");
}

}  // namespace

#ifndef MI_ELEM_F16
extern "C" size_t mi_attn_decode_workspace_bytes(int32_t batch, int32_t n_q_heads, int32_t head_dim, int32_t max_ctx) {
    (void)max_ctx;
    if (batch <= 0 || n_q_heads <= 0 || head_dim <= 0) return 0;
    return (size_t)batch * n_q_heads * kMaxSplits * (size_t)(head_dim + 2) * sizeof(float);
}
#endif

namespace {
// Validation and launches shared by the two entry points; `ws` / `ws_bytes` is the scratch for the per-split partial
// results (the caller's workspace, or the library's own static array for mi_attn_decode_static).
int decode_entry(const mi_decode_args* a, void* ws, size_t ws_bytes, bool static_ws, int32_t* tickets, int64_t n_tickets) {
    if (!a) return mi_fail(MI_E_NULL, "attn_decode: args is null");
    if (!a->q || !a->k_cache || !a->v_cache || !a->o || !a->ctx_len) return mi_fail(MI_E_NULL, "attn_decode: q, caches, o and ctx_len are required");
    if (a->dtype != MI_ELEM_DTYPE) return mi_fail(MI_E_DTYPE, "attn_decode: the decode kernels take bf16 or f16 tensors (dtype code %d)", a->dtype);
    if (a->head_dim != 32 && a->head_dim != 64 && a->head_dim != 96 && a->head_dim != 128)
        return mi_fail(MI_E_SHAPE, "attn_decode: head_dim %d unsupported (32, 64, 96, 128)", a->head_dim);
    if (a->batch <= 0 || a->max_ctx <= 0 || a->n_q_heads <= 0 || a->n_kv_heads <= 0 || a->n_q_heads % a->n_kv_heads != 0)
        return mi_fail(MI_E_SHAPE, "attn_decode: bad batch/head configuration");
    if ((a->k_new == nullptr) != (a->v_new == nullptr)) return mi_fail(MI_E_NULL, "attn_decode: k_new and v_new go together");
    const bool rot = a->rotary_cos != nullptr || a->rotary_sin != nullptr;
    if (rot && (!a->rotary_cos || !a->rotary_sin || !a->position_ids || a->rotary_table_rows <= 0))
        return mi_fail(MI_E_NULL, "attn_decode: fused rotary needs cos, sin, position ids and the table size");
    if (rot && !a->rotary_interleaved && a->head_dim != 64 && a->head_dim != 128)
        return mi_fail(MI_E_SHAPE, "attn_decode: fused rotate-half rotary needs head_dim 64 or 128");
    if (!mi_aligned16(a->q) || !mi_aligned16(a->k_cache) || !mi_aligned16(a->v_cache) || !mi_aligned16(a->o) ||
        (a->k_new && (!mi_aligned16(a->k_new) || !mi_aligned16(a->v_new))) ||
        (rot && (!mi_aligned16(a->rotary_cos) || !mi_aligned16(a->rotary_sin))))
        return mi_fail(MI_E_ALIGN, "attn_decode: tensors must be 16-byte aligned");
    if (a->cache_stride_batch % 8 || a->cache_stride_token % 8 || a->cache_stride_head % 8 || a->q_stride_batch % 8 ||
        a->k_new_stride_batch % 8 || a->v_new_stride_batch % 8)
        return mi_fail(MI_E_ALIGN, "attn_decode: strides must be multiples of 8 elements");
    if ((a->q_stride_batch && a->q_stride_batch < (int64_t)a->n_q_heads * a->head_dim) ||
        (a->k_new_stride_batch && a->k_new_stride_batch < (int64_t)a->n_kv_heads * a->head_dim) ||
        (a->v_new_stride_batch && a->v_new_stride_batch < (int64_t)a->n_kv_heads * a->head_dim))
        return mi_fail(MI_E_SHAPE, "attn_decode: a sequence stride is smaller than heads * head_dim");
    if (!(a->softmax_scale > 0.f)) return mi_fail(MI_E_SHAPE, "attn_decode: softmax_scale must be positive");
    const int n_hc = (a->n_q_heads / a->n_kv_heads + 15) / 16;
    int splits = a->n_splits > 0 ? a->n_splits : choose_splits(a->batch, a->n_kv_heads * n_hc, a->max_ctx);
    if (splits > kMaxSplits) splits = kMaxSplits;
    const size_t need = (size_t)a->batch * a->n_q_heads * splits * (size_t)(a->head_dim + 2) * sizeof(float);
    if (static_ws && need > ws_bytes)
        return mi_fail(MI_E_WORKSPACE, "attn_decode_static: batch %d x %d query heads x %d key splits x head_dim %d needs %zu bytes of "
                       "scratch, the library's static array holds %zu; use mi_attn_decode with a caller workspace",
                       a->batch, a->n_q_heads, splits, a->head_dim, need, ws_bytes);
    if (!ws || ws_bytes < need || !mi_aligned16(ws))
        return mi_fail(MI_E_WORKSPACE, "attn_decode: workspace needs %zu bytes (16-byte aligned), got %zu", need, ws_bytes);
    if (tickets && (n_tickets < (int64_t)a->batch * a->n_kv_heads * n_hc || (reinterpret_cast<uintptr_t>(tickets) & 3u) != 0))
        return mi_fail(MI_E_WORKSPACE, "attn_decode: %lld tickets (4-byte aligned), got %lld", (long long)a->batch * a->n_kv_heads * n_hc, (long long)n_tickets);
    DecodeParams p{};
    p.tickets = tickets;
    p.q = (const elem_t*)a->q; p.kc = (elem_t*)a->k_cache; p.vc = (elem_t*)a->v_cache; p.o = (elem_t*)a->o;
    p.ctx_len = a->ctx_len; p.k_new = (const elem_t*)a->k_new; p.v_new = (const elem_t*)a->v_new;
    if (a->rotary_interleaved) {
        p.cos32 = (const float*)a->rotary_cos; p.sin32 = (const float*)a->rotary_sin;
    } else {
        p.cos = (const elem_t*)a->rotary_cos; p.sin = (const elem_t*)a->rotary_sin;
    }
    p.pos = a->position_ids;
    p.table_rows = (int)a->rotary_table_rows;
    p.batch = a->batch; p.max_ctx = a->max_ctx; p.nq = a->n_q_heads; p.nkv = a->n_kv_heads;
    p.n_rep = a->n_q_heads / a->n_kv_heads; p.n_splits = splits; p.n_hc = n_hc;
    p.splits_m = divide_m(splits); p.groups_m = divide_m((uint32_t)(p.nkv * n_hc)); p.hc_m = divide_m(n_hc);
    p.c_sb = a->cache_stride_batch; p.c_st = a->cache_stride_token; p.c_sh = a->cache_stride_head;
    p.q_sb = a->q_stride_batch ? a->q_stride_batch : (int64_t)a->n_q_heads * a->head_dim;
    p.kn_sb = a->k_new_stride_batch ? a->k_new_stride_batch : (int64_t)a->n_kv_heads * a->head_dim;
    p.vn_sb = a->v_new_stride_batch ? a->v_new_stride_batch : (int64_t)a->n_kv_heads * a->head_dim;
    p.scale_log2 = a->softmax_scale * 1.4426950408889634f;
    if (p.tickets != nullptr && !merges_in_launch(p, a->head_dim)) p.tickets = nullptr;
    p.ws_o = (float*)ws;
    p.ws_ml = p.ws_o + (size_t)a->batch * a->n_q_heads * splits * a->head_dim;
    hipStream_t st = (hipStream_t)a->stream;
    const int rot_mode = rot ? (a->rotary_interleaved ? 2 : 1) : 0;
    switch (a->head_dim) {
        case 32: return launch_decode<32>(p, rot_mode, st);
        case 64: return launch_decode<64>(p, rot_mode, st);
        case 96: return launch_decode<96>(p, rot_mode, st);
        default: return launch_decode<128>(p, rot_mode, st);
    }
}
}  // namespace

int MI_ENTRY(mi_attn_decode_impl)(const mi_decode_args* a, bool static_ws, int32_t* tickets, int64_t n_tickets) {
    if (!a) return mi_fail(MI_E_NULL, "attn_decode: args is null");
    if (!static_ws) return decode_entry(a, a->workspace, a->workspace_bytes, false, tickets, n_tickets);
    // the entry point that allocates nothing: partial results go to the library's static device array
    void* ws = nullptr;
    size_t bytes = 0;
    const int rc = mi_static_scratch(&ws, &bytes);
    if (rc != MI_OK) return rc;
    return decode_entry(a, ws, bytes, true, nullptr, 0);
}
