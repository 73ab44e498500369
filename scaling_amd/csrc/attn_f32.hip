// Attention core for float32 tensors (the reference's default `precision`): forward, delta, dK/dV, dQ.
//
// Exact fp32 semantics of core/nn/attention/attention.py:108-213 with an fp32 tensor dtype: scores, softmax,
// probabilities and both products in fp32 (probs.to(value.dtype) is the identity), on the fp32 matrix pipe
// (v_mfma_f32_32x32x2_f32, 157 TFLOP/s class, a sixteenth of the bf16 rate).  Same masks, GQA index math, layouts,
// lse and workspace contract as the 16-bit kernels; no dropout and no fused rotary (rotate with mi_rotary /
// mi_rotary_complex first).
//
// v_mfma_f32_32x32x2_f32 operands, lane = 32 g + l32:  A: row l32, k = g;  B: column l32, k = g;
// C / D: column l32, rows 8 (r / 4) + 4 g + r % 4 for r = 0..15.  One such product takes 64 cycles of a SIMD, so the
// kernels are bound by the matrix pipe as long as its operands arrive, and what matters is that every SIMD always has
// products to issue:
//   * a workgroup is four wavefronts that stream tiles of 32 rows through LDS, loaded global -> LDS directly, one
//     step ahead of their use (one barrier per step);
//   * a contraction over features may visit them in any order, so lane half g takes features 8 j + 4 g .. + 3 of step j:
//     one 128-bit LDS read feeds four products;
//   * a C tile is reused as the B operand of the next product one register at a time (register r stands for the
//     contraction indices 8 (r / 4) + r % 4 and 4 more); the A operand is a row of the tile read along the features, and
//     output row l32 of tile dt stands for feature DT l32 + dt, so that one 128-bit read feeds all DT = 4 products of
//     head_dim 128 (64-bit for 64; head_dim 96 keeps 32 dt + l32);
//   * LDS rows are unpadded (a direct load writes 64 x 16 consecutive bytes); the 16-byte unit index of a row is XORed
//     with F32Tile::f(row), which spreads the 16 rows that one pass of a 128-bit read touches over all banks.
// One wavefront per workgroup with synchronous staging, the earlier form of these kernels, kept three of the four SIMDs
// of a compute unit busy at most and each of them waiting for its own loads: 19.1 ms for a forward + backward at 32 / 8
// heads of 128 and 4096 causal tokens (25 TFLOP/s).  With the backward as dK/dV and a dQ kernel that forms S and dP again 5.28 ms, 91 TFLOP/s (forward
// 1.08, delta 0.02, dK/dV 2.49, dQ 1.73 under the profiler, 5.33 together); where the products are a sixteenth of the 16-bit rate a byte of memory costs a
// sixteenth as much beside them, so dK/dV leaves dS in a workspace and dQ reads it: 4.24 ms, 113 TFLOP/s (dK/dV 2.60, dQ 0.58, 4.29 together).
#include "attn_common.h"

namespace {

constexpr float kLog2eF = 1.4426950408889634f;
constexpr int kF32Waves = 4;

__device__ __forceinline__ f32x16_t mfma_f32(float a, float b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// row index inside a 32-row tile that accumulator register r stands for in lane half g
__device__ __forceinline__ int acc_row(int r, int g) { return 8 * (r >> 2) + 4 * g + (r & 3); }

struct F32Params {
    const float* q; const float* k; const float* v; float* o; float* lse;
    const float* d_o; float* dq; float* dk; float* dv; float* delta;
    AttnParams m;     // masks, sizes, strides (the pointer members of m are not used)
    // backward, all of it in one call with room for dS: the dK/dV kernel leaves dS there and the dQ kernel reads it, for the KV heads
    // kv0 .. kv0 + kv_count - 1 at a time
    float* ds;
    int kv0, kv_count;
    bool ds_triangle;
};

// Where dS lies: tiles of 32 keys x 32 queries, [query head of the present KV heads][tile], each key's 32 queries contiguous.  Under a
// causal mask with the same documents on both axes no tile has its keys behind its queries, and the tiles form a triangle.
constexpr int kDsTile = 32 * 32;
inline bool ds_triangle(const mi_attn_args* a) {
    return a->causal && (a->cu_seqlens_k == nullptr || a->cu_seqlens_k == a->cu_seqlens_q) && a->total_q == a->total_k;
}
struct DsLayout {
    int64_t per_head;
    int k_tiles;                                           // 0: triangle
    __host__ __device__ DsLayout(int total_q, int total_k, bool triangle) {
        const int64_t nq = ((int64_t)total_q + 31) / 32, nk = ((int64_t)total_k + 31) / 32;
        per_head = triangle ? nq * (nq + 1) / 2 : nq * nk;
        k_tiles = triangle ? 0 : (int)nk;
    }
    __device__ __forceinline__ int64_t tile(int head, int q, int k) const {    // q, k: first token of the tile
        const int64_t i = q >> 5, j = k >> 5;
        return (head * per_head + (k_tiles == 0 ? i * (i + 1) / 2 : i * k_tiles) + j) * kDsTile;
    }
};

// ---- LDS tile of D floats per row ------------------------------------------------------------------------------------
template <int D> struct F32Tile {
    static constexpr int UPR = D / 4;         // 16-byte units per row
    static constexpr int RB = 4 * D;          // bytes per row
    static constexpr int DT = D / 32;
    // rows of 16 k units start on the same bank, rows of 8 and 24 units on two alternating ones
    static __device__ __forceinline__ int f(int r) { return UPR % 16 == 0 ? (r & 15) : ((r >> 1) & 7); }
    // feature of row `row` of output tile dt (see the header)
    static __device__ __forceinline__ int feature(int row, int dt) { return DT == 3 ? 32 * dt + row : DT * row + dt; }

    // features 8 j + 4 g .. + 3 of row `row`
    static __device__ __forceinline__ f32x4_t row4(const char* tile, int row, int j, int g) {
        return *reinterpret_cast<const f32x4_t*>(tile + row * RB + (((2 * j + g) ^ f(row)) << 4));
    }
    // the features of output row l32 in all DT tiles, taken from tile row `row`
    static __device__ __forceinline__ void cols(const char* tile, int row, int l32, float (&x)[DT]) {
        const char* base = tile + row * RB;
        if constexpr (DT == 4) {
            const f32x4_t v = *reinterpret_cast<const f32x4_t*>(base + ((l32 ^ f(row)) << 4));
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) x[dt] = v[dt];
        } else if constexpr (DT == 2) {
            const float2 v = *reinterpret_cast<const float2*>(base + (((l32 >> 1) ^ f(row)) << 4) + 8 * (l32 & 1));
            x[0] = v.x; x[1] = v.y;
        } else {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
                x[dt] = *reinterpret_cast<const float*>(base + (((8 * dt + (l32 >> 2)) ^ f(row)) << 4) + 4 * (l32 & 3));
        }
    }
};

// Direct global -> LDS loads of tiles of ROWS rows by the four wavefronts of a workgroup (see DmaPlan in attn_common.h
// for the reasons behind the inline assembly; completion is tracked with wait_vmcnt).
template <int D, int ROWS> struct F32Dma {
    using T = F32Tile<D>;
    static constexpr int kCount = ROWS * T::UPR / (64 * kF32Waves);   // instructions per wavefront
    static_assert(kCount >= 1 && ROWS * T::UPR % (64 * kF32Waves) == 0, "whole instructions");
    uint32_t off[kCount];
    int n0, lane;

    __device__ __forceinline__ static void src_of(int n, int lane_, int& row, int& byte) {
        const int u = 64 * n + lane_;
        row = u / T::UPR;
        byte = 16 * ((u % T::UPR) ^ T::f(row));
    }
    __device__ __forceinline__ void init(int wave, int lane_, int64_t row_stride) {
        n0 = wave * kCount;
        lane = lane_;
#pragma unroll
        for (int j = 0; j < kCount; ++j) {
            int row, byte;
            src_of(n0 + j, lane, row, byte);
            off[j] = (uint32_t)(row * (int)row_stride * 4 + byte);
        }
    }
    // instruction j of that alone, of a tile that is whole
    __device__ __forceinline__ void issue_whole(int j, const float* tile_base, char* tile) const {
        DmaPlan<D, 1>::issue_one(off[j], tile_base, tile + 1024 * (n0 + j));
    }
    // rows row0 .. row0 + ROWS - 1 of `base` (rows past last_row repeat it) into `tile`
    __device__ __forceinline__ void issue(const float* base, int64_t row_stride, int row0, int last_row, char* tile) const {
        char* dst = tile + 1024 * n0;
        const int first = min(row0, last_row);
        const float* tile_base = base + (int64_t)first * row_stride;
        if (row0 + ROWS - 1 <= last_row) {
#pragma unroll
            for (int j = 0; j < kCount; ++j) DmaPlan<D, 1>::issue_one(off[j], tile_base, dst + 1024 * j);
        } else {
            int l = lane;
            asm volatile("" : "+v"(l));   // opaque: keeps this rarely used arithmetic from being hoisted out of the caller's loop
#pragma unroll
            for (int j = 0; j < kCount; ++j) {
                int row, byte;
                src_of(n0 + j, l, row, byte);
                row = min(row, last_row - first);
                DmaPlan<D, 1>::issue_one((uint32_t)(row * (int)row_stride * 4 + byte), tile_base, dst + 1024 * j);
            }
        }
    }
};

// this lane's share of a row as the B operand of a contraction over features: features 8 j + 4 g .. + 3, j = 0 .. D/8 - 1
template <int D> __device__ __forceinline__ void load_operand(const float* row, int g, f32x4_t (&x)[D / 8]) {
#pragma unroll
    for (int j = 0; j < D / 8; ++j) x[j] = *reinterpret_cast<const f32x4_t*>(row + 8 * j + 4 * g);
    // consumed here: otherwise the loads count as possibly outstanding inside the tile loop
#pragma unroll
    for (int j = 0; j < D / 8; ++j) asm volatile("" : "+v"(x[j]));
}

// C = A B^T over the features: A rows row0 .. row0 + 31 of an LDS tile, B from registers
template <int D>
__device__ __forceinline__ f32x16_t rows_product(const char* tile, int row, int g, const f32x4_t (&b)[D / 8]) {
    f32x16_t c;
#pragma unroll
    for (int r = 0; r < 16; ++r) c[r] = 0.f;
    f32x4_t a[2];
    a[0] = F32Tile<D>::row4(tile, row, 0, g);
#pragma unroll
    for (int j = 0; j < D / 8; ++j) {
        if (j + 1 < D / 8) a[(j + 1) & 1] = F32Tile<D>::row4(tile, row, j + 1, g);
#pragma unroll
        for (int i = 0; i < 4; ++i) c = mfma_f32(a[j & 1][i], b[j][i], c);
    }
    return c;
}

// acc[dt] += columns(tile)^T x: contraction over the 32 rows of the tile from row0 on, x = a C tile register by register
template <int D>
__device__ __forceinline__ void cols_product(f32x16_t (&acc)[D / 32], const char* tile, int row0, const f32x16_t& x, int l32, int g) {
    constexpr int DT = D / 32;
    float a[2][DT];
    F32Tile<D>::cols(tile, row0 + acc_row(0, g), l32, a[0]);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        if (r + 1 < 16) F32Tile<D>::cols(tile, row0 + acc_row(r + 1, g), l32, a[(r + 1) & 1]);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) acc[dt] = mfma_f32(a[r & 1][dt], x[r], acc[dt]);
    }
}

// The two products of a kernel whose wavefronts have a SIMD each, with the rest of its work between them: between(j) behind every fourth product of rows
// and behind the DT products of a row of columns.  They are inline assembly because the compiler keeps the gradients' accumulators in vector registers otherwise
// and moves all of them to accumulation registers and back in every step; C tiles that vector instructions read are in vector registers.  What the compiler
// does not see then are waits between a product and whoever reads its result (18 states): between() may read the C tile of the stage before, `last`, which
// passes through an empty statement behind the first products of this stage (four, or DT, of 16 states each), so that no read of it moves in front of them; and
// the gradients pass through `settled` at the end.
__device__ __forceinline__ void mma_v(f32x16_t& c, float a, float b) { asm volatile("v_mfma_f32_32x32x2_f32 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b)); }
__device__ __forceinline__ void mma_v0(f32x16_t& c, float a, float b) { asm volatile("v_mfma_f32_32x32x2_f32 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b)); }
__device__ __forceinline__ void mma_acc(f32x16_t& c, float a, float b) { asm volatile("v_mfma_f32_32x32x2_f32 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b)); }
__device__ __forceinline__ void clear_acc(f32x16_t& c) {
#pragma unroll
    for (int r = 0; r < 16; ++r) c[r] = 0.f;
    asm volatile("" : "+a"(c));
}
struct NoTile {};
__device__ __forceinline__ void behind(f32x16_t& last) { asm volatile("" : "+v"(last)); }
__device__ __forceinline__ void behind(NoTile) {}
template <int DT> __device__ __forceinline__ void settled(f32x16_t (&x)[DT], f32x16_t (&y)[DT]) {
    asm volatile("s_nop 15\n\ts_nop 15" : "+a"(x[0]), "+a"(y[0]));
#pragma unroll
    for (int dt = 1; dt < DT; ++dt) asm volatile("" : "+a"(x[dt]), "+a"(y[dt]));
}

// a0, x0: the first operand, read ahead; then(): reads the one of the product behind this
template <int D, class Last, class F, class G>
__device__ __forceinline__ void rows_product_with(f32x16_t& c, const char* tile, int row, int g, const f32x4_t& a0, const f32x4_t (&b)[D / 8], Last&& last, F&& between,
                                                  G&& then) {
    f32x4_t a[2];
    a[0] = a0;
    static_for<D / 8>([&](auto j_c) {
        constexpr int j = decltype(j_c)::value;
        if constexpr (j + 1 < D / 8) a[(j + 1) & 1] = F32Tile<D>::row4(tile, row, j + 1, g);
        else then();
        __builtin_amdgcn_sched_barrier(0);
        static_for<4>([&](auto i_c) {
            constexpr int i = decltype(i_c)::value;
            if constexpr (j == 0 && i == 0) mma_v0(c, a[0][0], b[0][0]);
            else mma_v(c, a[j & 1][i], b[j][i]);
        });
        if constexpr (j == 0) behind(last);
        between(j_c);
        __builtin_amdgcn_sched_barrier(0);
    });
}

template <int D, class Last, class F, class G>
__device__ __forceinline__ void cols_product_with(f32x16_t (&acc)[D / 32], const char* tile, int row0, const float (&x0)[D / 32], const f32x16_t& x, int l32, int g,
                                                  Last&& last, F&& between, G&& then) {
    constexpr int DT = D / 32;
    float a[2][DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) a[0][dt] = x0[dt];
    static_for<16>([&](auto r_c) {
        constexpr int r = decltype(r_c)::value;
        if constexpr (r + 1 < 16) F32Tile<D>::cols(tile, row0 + acc_row(r + 1, g), l32, a[(r + 1) & 1]);
        else then();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) mma_acc(acc[dt], a[r & 1][dt], x[r]);
        if constexpr (r == 0) behind(last);
        between(r_c);
        __builtin_amdgcn_sched_barrier(0);
    });
}

// stores the features that accumulator registers r0 .. r0 + N - 1 hold of one token's row
template <int D, int N>
__device__ __forceinline__ void store_row(float* row, const f32x16_t (&acc)[D / 32], int r0, float scale, int g) {
    constexpr int DT = D / 32;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int r = r0 + i, fr = acc_row(r, g);
        if constexpr (DT == 4) {
            f32x4_t x;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) x[dt] = acc[dt][r] * scale;
            *reinterpret_cast<f32x4_t*>(row + 4 * fr) = x;
        } else if constexpr (DT == 2) {
            *reinterpret_cast<float2*>(row + 2 * fr) = make_float2(acc[0][r] * scale, acc[1][r] * scale);
        } else {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) row[F32Tile<D>::feature(fr, dt)] = acc[dt][r] * scale;
        }
    }
}

// Sum of the accumulators that the N wavefronts of a group hold for the same 32 tokens, in a fixed order; wavefront `part`
// stores registers part * 16 / N .. of the token's row.  `slot` is the group's LDS area (N x DT x 16 x 64 floats, free for
// use); all wavefronts of the workgroup call (two barriers).
template <int D, int N>
__device__ __forceinline__ void sum_and_store(f32x16_t (&acc)[D / 32], float* slot, int part, int lane, int g, float* row, bool live, float scale) {
    constexpr int DT = D / 32, R = 16 / N;
    if constexpr (N == 1) {
        if (live) store_row<D, 16>(row, acc, 0, scale, g);
    } else {
        __syncthreads();
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int r = 0; r < 16; ++r) slot[((part * DT + dt) * 16 + r) * 64 + lane] = acc[dt][r];
        __syncthreads();
        // the register index must be a constant, the part is not: one copy of the code per part
        static_for<N>([&](auto part_c) {
            constexpr int P = decltype(part_c)::value;
            if (part == P) {
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int i = 0; i < R; ++i) {
                        float s = slot[((0 * DT + dt) * 16 + P * R + i) * 64 + lane];
#pragma unroll
                        for (int n = 1; n < N; ++n) s += slot[((n * DT + dt) * 16 + P * R + i) * 64 + lane];
                        acc[dt][P * R + i] = s;
                    }
                if (live) store_row<D, R>(row, acc, P * R, scale, g);
            }
        });
    }
}

// first and one-past-last token of the union of the wavefronts' ranges (empty: 0, 0); one barrier
__device__ __forceinline__ void block_range(int wmin, int wmax, int wave, int lane, int* lds, int& bmin, int& bmax) {
    if (lane == 0) { lds[wave] = wmin; lds[kF32Waves + wave] = wmax; }
    __syncthreads();
    bmin = 0x7fffffff;
    bmax = 0;
#pragma unroll
    for (int w = 0; w < kF32Waves; ++w) { bmin = min(bmin, lds[w]); bmax = max(bmax, lds[kF32Waves + w]); }
    if (bmax <= bmin) { bmin = 0; bmax = 0; }
    bmin = __builtin_amdgcn_readfirstlane(bmin);
    bmax = __builtin_amdgcn_readfirstlane(bmax);
}

// LDS bytes and stages of a kernel that streams two tensors in steps of ROWS rows: two stages where both take at most 128 KB, however
// many workgroups that leaves a compute unit, else one
template <int D, int ROWS> constexpr int stage_bytes() { return 2 * ROWS * 4 * D; }
template <int D, int ROWS> constexpr int n_stages() { return 2 * stage_bytes<D, ROWS>() <= 128 * 1024 ? 2 : 1; }

// ---- forward: QG groups of 32 queries of one head, 4 / QG wavefronts per group that take different 32-key tiles of a
// step; S^T = K Q^T (lane = query), O^T += V^T P^T -----------------------------------------------------------------------
template <int D, int QG>
__global__ __launch_bounds__(64 * kF32Waves, 2) void attn_f32_fwd_kernel(const F32Params fp) {
    constexpr int DT = D / 32, KG = kF32Waves / QG, BN = 32 * KG, BM = 32 * QG;
    constexpr int NS = n_stages<D, BN>(), TILE = BN * 4 * D;
    __shared__ __attribute__((aligned(1024))) char smem[NS * 2 * TILE];
    __shared__ int range_lds[2 * kF32Waves];
    __shared__ float ml_lds[2][kF32Waves][32];
    const AttnParams& p = fp.m;
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qg = wave % QG, kg = wave / QG;
    const int nqb = (p.total_q + BM - 1) / BM;
    int head, rank;
    head_and_rank(blockIdx.x, p.nq, head, rank);
    const int qb = block_for_rank(rank, nqb, p.n_docs, 0, true);
    const int kvh = head / p.n_rep;
    const int tq = qb * BM + qg * 32 + l32;
    int klo, khi;
    key_range(p, tq, klo, khi);
    const int wmin = __builtin_amdgcn_readfirstlane(group_min<64>(khi > klo ? klo : 0x7fffffff));
    const int wmax = __builtin_amdgcn_readfirstlane(group_max<64>(khi > klo ? khi : 0));
    int bmin, bmax;
    block_range(wmin, wmax, wave, lane, range_lds, bmin, bmax);
    const int kt0 = bmin & ~31, n_steps = (bmax - kt0 + BN - 1) / BN;

    const float* kbase = fp.k + (int64_t)kvh * p.k_sh;
    const float* vbase = fp.v + (int64_t)kvh * p.v_sh;
    F32Dma<D, BN> k_dma, v_dma;
    k_dma.init(wave, lane, p.k_st);
    v_dma.init(wave, lane, p.v_st);
    auto issue = [&](int t) {
        if (t >= n_steps) return;
        char* st = smem + (t % NS) * 2 * TILE;
        k_dma.issue(kbase, p.k_st, kt0 + t * BN, p.total_k - 1, st);
        v_dma.issue(vbase, p.v_st, kt0 + t * BN, p.total_k - 1, st + TILE);
    };
    f32x4_t qf[D / 8];
    load_operand<D>(fp.q + (int64_t)min(tq, p.total_q - 1) * p.q_st + (int64_t)head * p.q_sh, g, qf);
    issue(0);
    f32x16_t o_acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o_acc[dt][r] = 0.f;
    float m_i = -INFINITY, l_i = 0.f;
    const float c2 = p.scale_log2;
    for (int t = 0; t < n_steps; ++t) {
        wait_vmcnt<0>();
        __syncthreads();                  // step t has landed, and the readers of step t - 1 are done
        if constexpr (NS == 2) issue(t + 1);
        const int kt = kt0 + t * BN + 32 * kg;
        if (kt < wmax && kt + 32 > wmin) {
            const char* k_s = smem + (t % NS) * 2 * TILE;
            const char* v_s = k_s + TILE;
            f32x16_t s = rows_product<D>(k_s, 32 * kg + l32, g, qf);        // rows = keys, column = this lane's query
            if (__any(kt < klo || kt + 32 > khi)) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int key = kt + acc_row(r, g);
                    if (key < klo || key >= khi) s[r] = -INFINITY;
                }
            }
            float mx = s[0];
#pragma unroll
            for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
            const float m_cand = pair_max(mx) * c2;
            if (__any(m_cand > m_i)) {    // rare after the first tiles: the accumulators are rescaled only then
                const float m_new = fmaxf(m_i, m_cand);
                float alpha = m_new == -INFINITY ? 1.0f : fast_exp2(m_i - m_new);
                asm volatile("" : "+v"(alpha));
                m_i = m_new;
                l_i *= alpha;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int r = 0; r < 16; ++r) o_acc[dt][r] *= alpha;
            }
            const float m_use = m_i == -INFINITY ? 0.f : m_i;
            float rs = 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                s[r] = fast_exp2(s[r] * c2 - m_use);
                rs += s[r];
            }
            l_i += rs;
            cols_product<D>(o_acc, v_s, 32 * kg, s, l32, g);
        }
        if constexpr (NS == 1) {
            __syncthreads();
            issue(t + 1);
        }
    }
    float l_tot = pair_sum(l_i), scale = 1.0f;
    if constexpr (KG > 1) {               // bring the partial results of the group's wavefronts to one maximum
        if (g == 0) { ml_lds[0][wave][l32] = m_i; ml_lds[1][wave][l32] = l_tot; }
        __syncthreads();
        float m_all = -INFINITY, l_all = 0.f;
#pragma unroll
        for (int n = 0; n < KG; ++n) m_all = fmaxf(m_all, ml_lds[0][n * QG + qg][l32]);
#pragma unroll
        for (int n = 0; n < KG; ++n) {
            const float m_n = ml_lds[0][n * QG + qg][l32];
            l_all += m_n == -INFINITY ? 0.f : ml_lds[1][n * QG + qg][l32] * fast_exp2(m_n - m_all);
        }
        scale = m_i == -INFINITY ? 0.f : fast_exp2(m_i - m_all);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int r = 0; r < 16; ++r) o_acc[dt][r] *= scale;
        m_i = m_all;
        l_tot = l_all;
    }
    const bool live = tq < p.total_q;
    float* slot = reinterpret_cast<float*>(smem) + (size_t)qg * KG * DT * 16 * 64;
    static_assert(QG * KG * DT * 16 * 64 * 4 <= NS * 2 * TILE || KG == 1, "the exchange reuses the tile stages");
    sum_and_store<D, KG>(o_acc, slot, kg, lane, g, fp.o + (int64_t)tq * p.o_st + (int64_t)head * p.o_sh, live, l_tot > 0.f ? 1.0f / l_tot : 0.f);
    if (live && kg == 0 && g == 0 && fp.lse != nullptr)
        fp.lse[(int64_t)head * p.total_q + tq] = l_tot > 0.f ? (m_i + __log2f(l_tot)) * 0.6931471805599453f : INFINITY;
}

// ---- delta[h][t] = sum_d dO[t][h][d] O[t][h][d] -----------------------------------------------------------------------
template <int D>
__global__ __launch_bounds__(256) void attn_f32_delta_kernel(const F32Params fp) {
    constexpr int LPR = D / 4;            // lanes per (token, head) row: 8, 16, 24 or 32
    constexpr int RPB = 256 / 32;         // rows per block: 32 lanes are reserved per row whatever D
    const AttnParams& p = fp.m;
    const int64_t row = (int64_t)blockIdx.x * RPB + threadIdx.x / 32;
    const int c = threadIdx.x % 32;
    const int64_t n_rows = (int64_t)p.total_q * p.nq;
    float acc = 0.f;
    const bool ok = row < n_rows && c < LPR;
    const int64_t t = row < n_rows ? row / p.nq : 0;
    const int h = row < n_rows ? (int)(row % p.nq) : 0;
    if (ok) {
        const f32x4_t a = *reinterpret_cast<const f32x4_t*>(fp.o + t * p.o_st + (int64_t)h * p.o_sh + 4 * c);
        const f32x4_t b = *reinterpret_cast<const f32x4_t*>(fp.d_o + t * p.o_st + (int64_t)h * p.o_sh + 4 * c);
        acc = a[0] * b[0] + a[1] * b[1] + a[2] * b[2] + a[3] * b[3];
    }
    acc = group_sum<32>(acc);
    if (row < n_rows && c == 0) fp.delta[(int64_t)h * p.total_q + t] = acc;
}

// ---- dK / dV: KGRP groups of 32 keys of one KV head (K, V rows in registers), 4 / KGRP wavefronts per group that take
// different 32-query tiles of a step; loops over the group's query heads and over the query steps: S = Q K^T, dP = dO V^T
// (lane = key), dV^T += dO^T P, dK^T += Q^T dS.  One wavefront per SIMD: K, V and both accumulators take 256 registers. ----
template <int D, int KGRP, bool KEEP>
__global__ __launch_bounds__(64 * kF32Waves, 1) void attn_f32_dkdv_kernel(const F32Params fp) {
    constexpr int DT = D / 32, QS = kF32Waves / KGRP, BQ = 32 * QS, BK = 32 * KGRP;
    constexpr int NS = n_stages<D, BQ>(), TILE = BQ * 4 * D;
    // A wavefront has its SIMD to itself and a product takes the matrix pipe 64 cycles, so loads, softmax and moves between two stages of a step cost what they
    // take: 0.68 of the pipe's rate at 2.4 GHz, 0.74 with all of them between products (busy 0.80 of a compute unit's cycles; the rest: a clock of 2.07 GHz instead of 2.17,
    // the barrier of a step, the last blocks of the launch).  us, before / after: 32 / 8 heads of 128, 4096 tokens 2600 / 2380, 32 / 32, 1101 245 / 230, 8 / 8, 700 (KGRP 1) 70.2 / 66.9; of 96, 32 / 32, 1101
    // 201 / 186.  Where stages are short or one tile deep it does not pay: of 96, KGRP 1 564 / 583, of 64, KGRP 1 100.0 / 101.1 and 11.1 / 11.7, of 32 358 / 359.
    constexpr bool kBetween = D == 128 || (D == 96 && KGRP == 2);
    static_assert(!kBetween || DT >= 2, "dS is formed one row of products behind dP");
    __shared__ __attribute__((aligned(1024))) char smem[NS * 2 * TILE];
    __shared__ __attribute__((aligned(16))) float lse_lds[2][BQ], delta_lds[2][BQ];
    __shared__ int range_lds[2 * kF32Waves];
    const AttnParams& p = fp.m;
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kgrp = wave % KGRP, qs = wave / KGRP;
    const int nkb = (p.total_k + BK - 1) / BK;
    // (KV head, split of its query heads) groups; the workgroup takes query heads kvh * n_rep + hs * hpw .. + hpw
    int group, rank;
    head_and_rank(blockIdx.x, (KEEP ? fp.kv_count : p.nkv) * p.hsplit, group, rank);
    const int first_kv = KEEP ? fp.kv0 : 0;
    const int kvh = first_kv + group / p.hsplit, hs = group - (kvh - first_kv) * p.hsplit, hpw = p.n_rep / p.hsplit;
    const int kb = block_for_rank(rank, nkb, p.n_docs, 0, false);
    const int key = kb * BK + kgrp * 32 + l32;
    int qlo, qhi;
    query_range(p, key, qlo, qhi);
    const int wmin = __builtin_amdgcn_readfirstlane(group_min<64>(qhi > qlo ? qlo : 0x7fffffff));
    const int wmax = __builtin_amdgcn_readfirstlane(group_max<64>(qhi > qlo ? qhi : 0));
    int bmin, bmax;
    block_range(wmin, wmax, wave, lane, range_lds, bmin, bmax);
    const int qt0 = bmin & ~31, n_tiles = (bmax - qt0 + BQ - 1) / BQ, n_steps = n_tiles * hpw;

    F32Dma<D, BQ> q_dma, do_dma;
    q_dma.init(wave, lane, p.q_st);
    do_dma.init(wave, lane, p.o_st);
    // (query head of the group, query tile) of the next step; heads outermost, in a fixed order: bit-reproducible sums
    int nxt_rep = 0, nxt_tile = 0, nxt = 0;
    // log-sum-exp and delta of a step's queries, straight into LDS like the tiles: a load into a register would make the compiler wait for the stores of dS
    // behind it as well
    auto issue_stat = [&](int head, int qt, int buf) {
        if (wave >= 2 * BQ / 64) return;
        const bool first = wave < BQ / 64;
        const int at = 64 * (first ? wave : wave - BQ / 64);
        const float* row = (first ? fp.lse : fp.delta) + (int64_t)head * p.total_q + qt;   // qt < total_q
        const uint32_t dst = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)(char*)((first ? lse_lds[buf] : delta_lds[buf]) + at);
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
                     ::"v"(4u * (uint32_t)min(at + lane, p.total_q - 1 - qt)), "s"(row), "s"(__builtin_amdgcn_readfirstlane(dst)) : "memory", "m0");
    };
    float stat = 0.f;                     // without kBetween they pass through a register of threads 0 .. 2 BQ - 1
    const float* stat_base = tid < BQ ? fp.lse : fp.delta;
    auto issue = [&]() {
        if (nxt >= n_steps) return;
        const int head = kvh * p.n_rep + hs * hpw + nxt_rep, qt = qt0 + nxt_tile * BQ;
        char* st = smem + (nxt % NS) * 2 * TILE;
        q_dma.issue(fp.q + (int64_t)head * p.q_sh, p.q_st, qt, p.total_q - 1, st);
        do_dma.issue(fp.d_o + (int64_t)head * p.o_sh, p.o_st, qt, p.total_q - 1, st + TILE);
        if constexpr (kBetween) issue_stat(head, qt, nxt & 1);
        else if (tid < 2 * BQ) stat = stat_base[(int64_t)head * p.total_q + min(qt + (tid & (BQ - 1)), p.total_q - 1)];
        if (++nxt_tile == n_tiles) { nxt_tile = 0; ++nxt_rep; }
        ++nxt;
    };
    auto put_stat = [&](int step) {
        if (tid < BQ) lse_lds[step & 1][tid] = stat * kLog2eF;
        else if (tid < 2 * BQ) delta_lds[step & 1][tid - BQ] = stat;
    };
    f32x4_t kf[D / 8], vf[D / 8];
    {
        const int kk = min(key, p.total_k - 1);
        load_operand<D>(fp.k + (int64_t)kk * p.k_st + (int64_t)kvh * p.k_sh, g, kf);
        load_operand<D>(fp.v + (int64_t)kk * p.v_st + (int64_t)kvh * p.v_sh, g, vf);
    }
    issue();
    f32x16_t dk_acc[DT], dv_acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
        if constexpr (kBetween) {
            clear_acc(dk_acc[dt]);
            clear_acc(dv_acc[dt]);
        } else {
#pragma unroll
            for (int r = 0; r < 16; ++r) { dk_acc[dt][r] = 0.f; dv_acc[dt][r] = 0.f; }
        }
    }
    const float c2 = p.scale_log2;
    const DsLayout ds(p.total_q, p.total_k, fp.ds_triangle);
    int tile = 0, rep = 0;
    if constexpr (kBetween) {
        // What is not a product goes between products: the direct loads of the next step between those of S, P between those of dP, dS between those of dV.
        constexpr int kLoads = F32Dma<D, BQ>::kCount, kParts = D / 8;
        bool stored = false;                  // by the step before, behind its loads: four stores that need not have arrived
        for (int step = 0; step < n_steps; ++step) {
            if (KEEP && NS == 2 && stored) wait_vmcnt<4>(); else wait_vmcnt<0>();
            __syncthreads();                  // the step has landed, and the readers of the one before are done
            const int qt = qt0 + tile * BQ + 32 * qs, head = kvh * p.n_rep + hs * hpw + rep;
            if (++tile == n_tiles) { tile = 0; ++rep; }
            const bool wanted = qt < wmax && qt + 32 > wmin;
            // the next step's tiles, if they are whole: as issue() requests them
            const int next_qt = qt0 + nxt_tile * BQ, next_head = kvh * p.n_rep + hs * hpw + nxt_rep;
            const bool between = NS == 2 && wanted && nxt < n_steps && next_qt + BQ <= p.total_q;
            const float* next_q = fp.q + (int64_t)next_head * p.q_sh + (int64_t)next_qt * p.q_st;
            const float* next_do = fp.d_o + (int64_t)next_head * p.o_sh + (int64_t)next_qt * p.o_st;
            char* next_stage = smem + (nxt % NS) * 2 * TILE;
            if (between) {
                issue_stat(next_head, next_qt, nxt & 1);
                if (++nxt_tile == n_tiles) { nxt_tile = 0; ++nxt_rep; }
                ++nxt;
            } else if constexpr (NS == 2) {
                issue();
            }
            stored = wanted;
            if (wanted) {
                const char* q_s = smem + (step % NS) * 2 * TILE;
                const char* do_s = q_s + TILE;
                int l = l32, h = g;
                asm volatile("" : "+v"(l), "+v"(h));   // opaque: the swizzled LDS addresses are made where they are used, not kept in registers over the steps
                f32x16_t s, dp;                   // rows = queries, column = this lane's key
                f32x4_t row0;
                float col0[2][DT];
                rows_product_with<D>(s, q_s, 32 * qs + l, h, F32Tile<D>::row4(q_s, 32 * qs + l, 0, h), kf, NoTile{}, [&](auto j) {
                    if (between) {
                        static_for<2 * kLoads>([&](auto n_c) {
                            constexpr int n = decltype(n_c)::value;
                            if constexpr (n * kParts / (2 * kLoads) == decltype(j)::value) {
                                if constexpr (n < kLoads) q_dma.issue_whole(n, next_q, next_stage);
                                else do_dma.issue_whole(n - kLoads, next_do, next_stage + TILE);
                            }
                        });
                    }
                }, [&] { row0 = F32Tile<D>::row4(do_s, 32 * qs + l, 0, h); });
                const unsigned seen = (unsigned)(qhi - qlo);
                const int rel0 = qt + 4 * h - qlo;
                const float* lse_row = &lse_lds[step & 1][32 * qs + 4 * h];
                const float* delta_row = &delta_lds[step & 1][32 * qs + 4 * h];
                auto log2_sums = [&](int a) {     // rounded before they are subtracted, as a product of their own
                    f32x4_t l4 = *reinterpret_cast<const f32x4_t*>(lse_row + 8 * a) * kLog2eF;
                    asm volatile("" : "+v"(l4));
                    return l4;
                };
                f32x4_t l4 = log2_sums(0);
                rows_product_with<D>(dp, do_s, 32 * qs + l, h, row0, vf, s, [&](auto j) {
                    static_for<16>([&](auto r_c) {
                        constexpr int r = decltype(r_c)::value, a = r >> 2, c = r & 3;
                        if constexpr (r * kParts / 16 == decltype(j)::value) {
                            float pv = fast_exp2(s[r] * c2 - l4[c]);
                            pv = (unsigned)(rel0 + 8 * a + c) < seen ? pv : 0.f;
                            asm volatile("" : "+v"(pv));   // here, not where it is used
                            s[r] = pv;
                            if constexpr (c == 3 && a < 3) l4 = log2_sums(a + 1);
                        }
                    });
                }, [&] { F32Tile<D>::cols(do_s, 32 * qs + acc_row(0, h), l, col0[0]); });
                f32x4_t d4 = *reinterpret_cast<const f32x4_t*>(delta_row);
                float* out = KEEP ? fp.ds + ds.tile(head - first_kv * p.n_rep, qt, kb * BK + kgrp * 32) + l32 * 32 + 4 * g : nullptr;
                cols_product_with<D>(dv_acc, do_s, 32 * qs, col0[0], s, l, h, dp, [&](auto r_c) {
                    constexpr int r = decltype(r_c)::value, a = r >> 2, c = r & 3;
                    float dsv = s[r] * (dp[r] - d4[c]);
                    asm volatile("" : "+v"(dsv));
                    dp[r] = dsv;
                    if constexpr (c == 3) {
                        if constexpr (KEEP) *reinterpret_cast<f32x4_t*>(out + 8 * a) = f32x4_t{dp[4 * a], dp[4 * a + 1], dp[4 * a + 2], dp[4 * a + 3]};
                        if constexpr (a < 3) d4 = *reinterpret_cast<const f32x4_t*>(delta_row + 8 * (a + 1));
                    }
                }, [&] { F32Tile<D>::cols(q_s, 32 * qs + acc_row(0, h), l, col0[1]); });
                cols_product_with<D>(dk_acc, q_s, 32 * qs, col0[1], dp, l, h, NoTile{}, [](auto) {}, [] {});
            }
            if constexpr (NS == 1) {
                __syncthreads();
                issue();
            }
        }
        settled(dk_acc, dv_acc);
    } else {
        for (int step = 0; step < n_steps; ++step) {
            put_stat(step);
            wait_vmcnt<0>();
            __syncthreads();                  // the step has landed, and the readers of the one before are done
            if constexpr (NS == 2) issue();
            const int qt = qt0 + tile * BQ + 32 * qs, head = kvh * p.n_rep + hs * hpw + rep;
            if (++tile == n_tiles) { tile = 0; ++rep; }
            if (qt < wmax && qt + 32 > wmin) {
                const char* q_s = smem + (step % NS) * 2 * TILE;
                const char* do_s = q_s + TILE;
                f32x16_t s = rows_product<D>(q_s, 32 * qs + l32, g, kf);         // rows = queries, column = this lane's key
                f32x16_t dp = rows_product<D>(do_s, 32 * qs + l32, g, vf);
                const bool edge = __any(qt < qlo || qt + 32 > qhi);
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    const f32x4_t l4 = *reinterpret_cast<const f32x4_t*>(&lse_lds[step & 1][32 * qs + 8 * a + 4 * g]);
                    const f32x4_t d4 = *reinterpret_cast<const f32x4_t*>(&delta_lds[step & 1][32 * qs + 8 * a + 4 * g]);
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const int r = 4 * a + c;
                        float pv = fast_exp2(s[r] * c2 - l4[c]);
                        if (edge) {
                            const int q = qt + 8 * a + 4 * g + c;
                            if (q < qlo || q >= qhi) pv = 0.f;
                        }
                        s[r] = pv;
                        dp[r] = pv * (dp[r] - d4[c]);
                    }
                }
                if constexpr (KEEP) {
                    float* out = fp.ds + ds.tile(head - first_kv * p.n_rep, qt, kb * BK + kgrp * 32) + l32 * 32 + 4 * g;
#pragma unroll
                    for (int a = 0; a < 4; ++a) *reinterpret_cast<f32x4_t*>(out + 8 * a) = f32x4_t{dp[4 * a], dp[4 * a + 1], dp[4 * a + 2], dp[4 * a + 3]};
                }
                cols_product<D>(dv_acc, do_s, 32 * qs, s, l32, g);
                cols_product<D>(dk_acc, q_s, 32 * qs, dp, l32, g);
            }
            if constexpr (NS == 1) {
                __syncthreads();
                issue();
            }
        }
    }
    const bool live = key < p.total_k;
    float* slot = reinterpret_cast<float*>(smem) + (size_t)kgrp * QS * DT * 16 * 64;
    static_assert(KGRP * QS * DT * 16 * 64 * 4 <= NS * 2 * TILE || QS == 1, "the exchange reuses the tile stages");
    float* dk_row = fp.dk + (int64_t)key * p.dk_st + (int64_t)kvh * p.dk_sh;
    float* dv_row = fp.dv + (int64_t)key * p.dv_st + (int64_t)kvh * p.dv_sh;
    if (p.hsplit > 1) {
        const int64_t off = (((int64_t)hs * p.total_k + key) * p.nkv + kvh) * D;
        dk_row = p.dk_part + off;
        dv_row = p.dv_part + off;
    }
    sum_and_store<D, QS>(dk_acc, slot, qs, lane, g, dk_row, live, p.scale);
    sum_and_store<D, QS>(dv_acc, slot, qs, lane, g, dv_row, live, 1.0f);
}

// sum of the hsplit partial dK / dV rows of a split launch, in a fixed order; one thread per four features
template <int D>
__global__ __launch_bounds__(256) void attn_f32_dkdv_reduce_kernel(const F32Params fp) {
    const AttnParams& p = fp.m;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x, n = (int64_t)p.total_k * p.nkv * (D / 4);
    if (idx >= n) return;
    const int c = (int)(idx % (D / 4)), kvh = (int)((idx / (D / 4)) % p.nkv);
    const int64_t key = idx / ((int64_t)(D / 4) * p.nkv), stride = (int64_t)p.total_k * p.nkv * D;
    f32x4_t k4 = *reinterpret_cast<const f32x4_t*>(p.dk_part + 4 * idx), v4 = *reinterpret_cast<const f32x4_t*>(p.dv_part + 4 * idx);
    for (int s = 1; s < p.hsplit; ++s) {
        k4 += *reinterpret_cast<const f32x4_t*>(p.dk_part + s * stride + 4 * idx);
        v4 += *reinterpret_cast<const f32x4_t*>(p.dv_part + s * stride + 4 * idx);
    }
    *reinterpret_cast<f32x4_t*>(fp.dk + key * p.dk_st + (int64_t)kvh * p.dk_sh + 4 * c) = k4;
    *reinterpret_cast<f32x4_t*>(fp.dv + key * p.dv_st + (int64_t)kvh * p.dv_sh + 4 * c) = v4;
}

// ---- dQ: QG groups of 32 queries of one head, 4 / QG wavefronts per group that take different 32-key tiles of a step:
// S^T = K Q^T, dP^T = V dO^T (lane = query), dQ^T += K^T dS^T.  head_dim 128: Q, dO and dQ take 192 registers, so one
// wavefront per SIMD (two, with 58 registers spilled: 2.1 against 1.8 ms at 4096 tokens of 32 / 8 heads) ----
template <int D, int QG>
__global__ __launch_bounds__(64 * kF32Waves, D == 128 ? 1 : 2) void attn_f32_dq_kernel(const F32Params fp) {
    constexpr int DT = D / 32, KG = kF32Waves / QG, BN = 32 * KG, BM = 32 * QG;
    constexpr int NS = n_stages<D, BN>(), TILE = BN * 4 * D;
    __shared__ __attribute__((aligned(1024))) char smem[NS * 2 * TILE];
    __shared__ int range_lds[2 * kF32Waves];
    const AttnParams& p = fp.m;
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qg = wave % QG, kg = wave / QG;
    const int nqb = (p.total_q + BM - 1) / BM;
    int head, rank;
    head_and_rank(blockIdx.x, p.nq, head, rank);
    const int qb = block_for_rank(rank, nqb, p.n_docs, 0, true);
    const int kvh = head / p.n_rep;
    const int tq = qb * BM + qg * 32 + l32;
    int klo, khi;
    key_range(p, tq, klo, khi);
    const int wmin = __builtin_amdgcn_readfirstlane(group_min<64>(khi > klo ? klo : 0x7fffffff));
    const int wmax = __builtin_amdgcn_readfirstlane(group_max<64>(khi > klo ? khi : 0));
    int bmin, bmax;
    block_range(wmin, wmax, wave, lane, range_lds, bmin, bmax);
    const int kt0 = bmin & ~31, n_steps = (bmax - kt0 + BN - 1) / BN;

    const float* kbase = fp.k + (int64_t)kvh * p.k_sh;
    const float* vbase = fp.v + (int64_t)kvh * p.v_sh;
    F32Dma<D, BN> k_dma, v_dma;
    k_dma.init(wave, lane, p.k_st);
    v_dma.init(wave, lane, p.v_st);
    auto issue = [&](int t) {
        if (t >= n_steps) return;
        char* st = smem + (t % NS) * 2 * TILE;
        k_dma.issue(kbase, p.k_st, kt0 + t * BN, p.total_k - 1, st);
        v_dma.issue(vbase, p.v_st, kt0 + t * BN, p.total_k - 1, st + TILE);
    };
    const int tl = min(tq, p.total_q - 1);
    f32x4_t qf[D / 8], dof[D / 8];
    load_operand<D>(fp.q + (int64_t)tl * p.q_st + (int64_t)head * p.q_sh, g, qf);
    load_operand<D>(fp.d_o + (int64_t)tl * p.o_st + (int64_t)head * p.o_sh, g, dof);
    float lse2 = fp.lse[(int64_t)head * p.total_q + tl] * kLog2eF;
    float delta = fp.delta[(int64_t)head * p.total_q + tl];
    asm volatile("" : "+v"(lse2), "+v"(delta));
    issue(0);
    f32x16_t dq_acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) dq_acc[dt][r] = 0.f;
    const float c2 = p.scale_log2;
    for (int t = 0; t < n_steps; ++t) {
        wait_vmcnt<0>();
        __syncthreads();
        if constexpr (NS == 2) issue(t + 1);
        const int kt = kt0 + t * BN + 32 * kg;
        if (kt < wmax && kt + 32 > wmin) {
            const char* k_s = smem + (t % NS) * 2 * TILE;
            const char* v_s = k_s + TILE;
            f32x16_t s = rows_product<D>(k_s, 32 * kg + l32, g, qf);            // rows = keys, column = this lane's query
            f32x16_t dp = rows_product<D>(v_s, 32 * kg + l32, g, dof);
            const bool edge = __any(kt < klo || kt + 32 > khi);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                float pv = fast_exp2(s[r] * c2 - lse2);
                if (edge) {
                    const int key = kt + acc_row(r, g);
                    if (key < klo || key >= khi) pv = 0.f;
                }
                dp[r] = pv * (dp[r] - delta);
            }
            cols_product<D>(dq_acc, k_s, 32 * kg, dp, l32, g);
        }
        if constexpr (NS == 1) {
            __syncthreads();
            issue(t + 1);
        }
    }
    float* slot = reinterpret_cast<float*>(smem) + (size_t)qg * KG * DT * 16 * 64;
    static_assert(QG * KG * DT * 16 * 64 * 4 <= NS * 2 * TILE || KG == 1, "the exchange reuses the tile stages");
    sum_and_store<D, KG>(dq_acc, slot, kg, lane, g, fp.dq + (int64_t)tq * p.q_st + (int64_t)head * p.q_sh, tq < p.total_q, p.scale);
}

// ---- dQ from the dS that the dK/dV kernel left: one product instead of three.  The key tiles of a step as above, the dS of the next one in
// registers: lane = query, one 128-byte line per key and half.  What no query may see was not written, or not by this call, and counts as zero. ----
template <int D, int QG>
__global__ __launch_bounds__(64 * kF32Waves, 2) void attn_f32_dq_kept_kernel(const F32Params fp) {
    constexpr int DT = D / 32, KG = kF32Waves / QG, BN = 32 * KG, BM = 32 * QG;
    constexpr int NS = 2, TILE = BN * 4 * D;
    __shared__ __attribute__((aligned(1024))) char smem[NS * TILE];
    __shared__ int range_lds[2 * kF32Waves];
    const AttnParams& p = fp.m;
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qg = wave % QG, kg = wave / QG;
    const int nqb = (p.total_q + BM - 1) / BM;
    int head, rank;
    head_and_rank(blockIdx.x, fp.kv_count * p.n_rep, head, rank);
    const int qb = block_for_rank(rank, nqb, p.n_docs, 0, true);
    const int kvh = fp.kv0 + head / p.n_rep;
    const int q0 = qb * BM + qg * 32, tq = q0 + l32;
    int klo, khi;
    key_range(p, tq, klo, khi);
    const int wmin = __builtin_amdgcn_readfirstlane(group_min<64>(khi > klo ? klo : 0x7fffffff));
    const int wmax = __builtin_amdgcn_readfirstlane(group_max<64>(khi > klo ? khi : 0));
    int bmin, bmax;
    block_range(wmin, wmax, wave, lane, range_lds, bmin, bmax);
    const int kt0 = bmin & ~31, n_steps = (bmax - kt0 + BN - 1) / BN;
    const float* kbase = fp.k + (int64_t)kvh * p.k_sh;
    F32Dma<D, BN> k_dma;
    k_dma.init(wave, lane, p.k_st);
    const float* ds = fp.ds + DsLayout(p.total_q, p.total_k, fp.ds_triangle).tile(head, q0, 0) + l32;
    f32x16_t next;
    auto issue = [&](int t) {
        if (t >= n_steps) return;
        const int kt = kt0 + t * BN + 32 * kg;
        if (kt < wmax && kt + 32 > wmin) {
            const float* from = ds + (int64_t)(kt >> 5) * kDsTile;
#pragma unroll
            for (int r = 0; r < 16; ++r) next[r] = from[acc_row(r, g) * 32];
        }
        k_dma.issue(kbase, p.k_st, kt0 + t * BN, p.total_k - 1, smem + (t % NS) * TILE);
    };
#pragma unroll
    for (int r = 0; r < 16; ++r) next[r] = 0.f;
    issue(0);
    f32x16_t dq_acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) dq_acc[dt][r] = 0.f;
    for (int t = 0; t < n_steps; ++t) {
        wait_vmcnt<0>();
        f32x16_t x = next;
        asm volatile("" : "+v"(x));           // arrived: the loads below are not waited for
        __syncthreads();
        issue(t + 1);
        const int kt = kt0 + t * BN + 32 * kg;
        if (kt < wmax && kt + 32 > wmin) {
            if (__any(kt < klo || kt + 32 > khi)) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int key = kt + acc_row(r, g);
                    if (key < klo || key >= khi) x[r] = 0.f;
                }
            }
            cols_product<D>(dq_acc, smem + (t % NS) * TILE, 32 * kg, x, l32, g);
        }
    }
    float* slot = reinterpret_cast<float*>(smem) + (size_t)qg * KG * DT * 16 * 64;
    static_assert(QG * KG * DT * 16 * 64 * 4 <= NS * TILE || KG == 1, "the exchange reuses the tile stages");
    sum_and_store<D, KG>(dq_acc, slot, kg, lane, g, fp.dq + (int64_t)tq * p.q_st + (int64_t)(fp.kv0 * p.n_rep + head) * p.q_sh, tq < p.total_q, p.scale);
}

int validate_f32(const mi_attn_args* a, const char* who) {
    int rc = mi_attn_validate(a, who, MI_F32, 4);
    if (rc != MI_OK) return rc;
    if (a->rotary_cos || a->rotary_sin) return mi_fail(MI_E_DTYPE, "%s: the fused rotary takes bf16 / f16 tensors; rotate fp32 q and k with mi_rotary first", who);
    if (a->dropout_p > 0.f) return mi_fail(MI_E_DTYPE, "%s: attention-probability dropout takes bf16 / f16 tensors", who);
    return MI_OK;
}

void fill(const mi_attn_args* a, F32Params* fp) {
    *fp = F32Params{};
    mi_attn_fill_params(a, &fp->m);
    fp->q = (const float*)a->q; fp->k = (const float*)a->k; fp->v = (const float*)a->v;
    fp->o = (float*)a->o; fp->lse = a->lse;
}

// Four query groups per workgroup (every staged K / V tile feeds four wavefronts) once that gives two workgroups per compute
// unit; below that, one query group whose four wavefronts split the keys.  Measured (head_dim 128, four groups / one):
// 512 blocks of 128 queries 385 / 407 us, 256 blocks 277 / 208 us, 16 blocks 39 / 17 us.
template <int D> int launch_fwd_f32(const F32Params& fp, hipStream_t st) {
    const AttnParams& p = fp.m;
    const dim3 block(64 * kF32Waves);
    const int64_t wide = (((int64_t)p.total_q + 127) / 128) * p.nq, narrow = (((int64_t)p.total_q + 31) / 32) * p.nq;
    if (wide >= 2 * mi_compute_units()) attn_f32_fwd_kernel<D, 4><<<dim3((unsigned)wide), block, 0, st>>>(fp);
    else attn_f32_fwd_kernel<D, 1><<<dim3((unsigned)narrow), block, 0, st>>>(fp);
    return mi_check_launch("attn_fwd (f32)");
}

}  // namespace

int mi_attn_fwd_impl_f32(const mi_attn_args* a) {
    int rc = validate_f32(a, "attn_fwd");
    if (rc != MI_OK) return rc;
    if (!a->o) return mi_fail(MI_E_NULL, "attn_fwd: o is null");
    if (!mi_aligned16(a->o) || a->o_stride_token % 4 || a->o_stride_head % 4)
        return mi_fail(MI_E_ALIGN, "attn_fwd: o must be 16-byte aligned with strides multiple of 4");
    if (a->total_q == 0) return MI_OK;
    F32Params fp;
    fill(a, &fp);
    if (((a->total_q + 31) / 32) * a->n_q_heads > 0x7fffffffLL) return mi_fail(MI_E_SHAPE, "attn_fwd: too many work items");
    hipStream_t st = (hipStream_t)a->stream;
    switch (a->head_dim) {
        case 32: return launch_fwd_f32<32>(fp, st);
        case 64: return launch_fwd_f32<64>(fp, st);
        case 96: return launch_fwd_f32<96>(fp, st);
        case 128: return launch_fwd_f32<128>(fp, st);
        default: return mi_fail(MI_E_SHAPE, "attn_fwd: head_dim %d unsupported (32, 64, 96, 128)", a->head_dim);
    }
}

// Backward with dS kept: five products instead of seven, the same bits.  Bytes of dS are bounded; what does not fit at once goes a number of
// KV heads at a time, each of them two workgroups per compute unit.  us, recomputed / kept (query heads / KV heads, head_dim, causal unless said):
//   32/32  64  1101 tokens  258 / 191     32/32 128  1101  443 / 336     12/12 128  14 x 300  334 / 252     16/16 128  8192  8199 / 6628 (2 passes)
//   16/16  64  8192        4310 / 3658    32/8  128  4096 4221 / 3167    32/32  64  64 x 64   167 / 131     32/32  64  1100, not causal  489 / 361
// At head_dim 32 the products that are saved take less time than the bytes.
static constexpr int64_t kDsBytes = (int64_t)5 << 28;             // 1.25 GiB

// KV heads per pass, 0: not at all
static int ds_heads(const mi_attn_args* a) {
    if (a->head_dim < 64 || a->total_q <= 0 || a->total_k <= 0 || a->n_kv_heads <= 0 || a->n_q_heads % a->n_kv_heads != 0 || a->total_q > 0x7fffff00LL ||
        a->total_k > 0x7fffff00LL)
        return 0;
    const DsLayout l((int)a->total_q, (int)a->total_k, ds_triangle(a));
    const int64_t each = l.per_head * kDsTile * (int64_t)sizeof(float) * (a->n_q_heads / a->n_kv_heads), fit = kDsBytes / each;
    if (fit < 1) return 0;
    const int passes = (int)((a->n_kv_heads + fit - 1) / fit), heads = (a->n_kv_heads + passes - 1) / passes;
    const int64_t blocks = (a->total_k + 63) / 64 * heads * mi_dkdv_head_split(a->n_q_heads, a->n_kv_heads);
    return blocks >= 2 * mi_compute_units() ? heads : 0;
}

template <int D> static int launch_reduce_f32(const F32Params& fp, hipStream_t st) {
    const AttnParams& p = fp.m;
    if (p.hsplit == 1) return MI_OK;
    const int64_t n = (int64_t)p.total_k * p.nkv * (D / 4);
    attn_f32_dkdv_reduce_kernel<D><<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st>>>(fp);
    return mi_check_launch("attn_bwd_dkdv_reduce (f32)");
}

template <int D> static int launch_kept_f32(const F32Params& all, hipStream_t st) {
    if constexpr (D < 64) return mi_fail(MI_E_SHAPE, "attn_bwd: dS is not kept at head_dim %d", D);
    else {
        F32Params fp = all;
        const AttnParams& p = fp.m;
        const dim3 block(64 * kF32Waves);
        const int step = all.kv_count;
        for (fp.kv0 = 0; fp.kv0 < p.nkv; fp.kv0 += step) {
            fp.kv_count = step < p.nkv - fp.kv0 ? step : p.nkv - fp.kv0;
            const int64_t keys = (((int64_t)p.total_k + 63) / 64) * fp.kv_count * p.hsplit, heads = (int64_t)fp.kv_count * p.n_rep;
            attn_f32_dkdv_kernel<D, 2, true><<<dim3((unsigned)keys), block, 0, st>>>(fp);
            int rc = mi_check_launch("attn_bwd_dkdv (f32)");
            if (rc != MI_OK) return rc;
            // by all heads, as where dS is not kept: the split of the keys is the order of the sums, which the room for dS must not decide
            const int64_t wide = (((int64_t)p.total_q + 127) / 128) * heads, narrow = (((int64_t)p.total_q + 31) / 32) * heads;
            if (wide / heads * p.nq >= 2 * mi_compute_units()) attn_f32_dq_kept_kernel<D, 4><<<dim3((unsigned)wide), block, 0, st>>>(fp);
            else attn_f32_dq_kept_kernel<D, 1><<<dim3((unsigned)narrow), block, 0, st>>>(fp);
            rc = mi_check_launch("attn_bwd_dq (f32)");
            if (rc != MI_OK) return rc;
        }
        return launch_reduce_f32<D>(fp, st);
    }
}

template <int D> static int launch_bwd_f32(const F32Params& fp, int flags, hipStream_t st) {
    const AttnParams& p = fp.m;
    const int stages = flags & (MI_ATTN_BWD_DELTA | MI_ATTN_BWD_DKDV | MI_ATTN_BWD_DQ);
    const bool all = stages == 0;
    const dim3 block(64 * kF32Waves);
    if (all || (stages & MI_ATTN_BWD_DELTA)) {
        const int64_t rows = (int64_t)p.total_q * p.nq;
        attn_f32_delta_kernel<D><<<dim3((unsigned)((rows + 7) / 8)), dim3(256), 0, st>>>(fp);
        int rc = mi_check_launch("attn_bwd_delta (f32)");
        if (rc != MI_OK) return rc;
    }
    if (all || (stages & MI_ATTN_BWD_DKDV)) {
        // two key groups per workgroup (each staged Q / dO tile feeds two wavefronts) from two workgroups per compute unit
        // on, which a causal mask needs to pair long key blocks with short ones; below that, one key group whose four
        // wavefronts split the queries.  Measured (head_dim 128, two groups / one): 512 blocks of 64 keys 331 / 377 us,
        // 384 blocks 1751 / 1656 us, 256 blocks 1168 / 700 us
        if (all && fp.ds != nullptr) return launch_kept_f32<D>(fp, st);
        const int64_t groups = (int64_t)p.nkv * p.hsplit;
        const int64_t wide = (((int64_t)p.total_k + 63) / 64) * groups, narrow = (((int64_t)p.total_k + 31) / 32) * groups;
        if (wide >= 2 * mi_compute_units()) attn_f32_dkdv_kernel<D, 2, false><<<dim3((unsigned)wide), block, 0, st>>>(fp);
        else attn_f32_dkdv_kernel<D, 1, false><<<dim3((unsigned)narrow), block, 0, st>>>(fp);
        int rc = mi_check_launch("attn_bwd_dkdv (f32)");
        if (rc != MI_OK) return rc;
        rc = launch_reduce_f32<D>(fp, st);
        if (rc != MI_OK) return rc;
    }
    if (all || (stages & MI_ATTN_BWD_DQ)) {
        const int64_t wide = (((int64_t)p.total_q + 127) / 128) * p.nq, narrow = (((int64_t)p.total_q + 31) / 32) * p.nq;
        // as for the forward (512 blocks of 128 queries 450 / 553 us, 256 blocks 414 / 278 us at head_dim 128)
        if (wide >= 2 * mi_compute_units()) attn_f32_dq_kernel<D, 4><<<dim3((unsigned)wide), block, 0, st>>>(fp);
        else attn_f32_dq_kernel<D, 1><<<dim3((unsigned)narrow), block, 0, st>>>(fp);
        return mi_check_launch("attn_bwd_dq (f32)");
    }
    return MI_OK;
}

size_t mi_attn_bwd_workspace_bytes_f32(const mi_attn_args* a) {
    const int heads = ds_heads(a);
    if (heads == 0) return 0;
    const DsLayout l((int)a->total_q, (int)a->total_k, ds_triangle(a));
    const size_t base = mi_attn_bwd_workspace_bytes_kv(a->total_q, a->total_k, a->n_q_heads, a->n_kv_heads, a->head_dim);
    return (base + 255) / 256 * 256 + (size_t)l.per_head * kDsTile * sizeof(float) * heads * (a->n_q_heads / a->n_kv_heads);
}

int mi_attn_bwd_impl_f32(const mi_attn_bwd_args* b) {
    if (!b) return mi_fail(MI_E_NULL, "attn_bwd: args is null");
    const mi_attn_args* a = &b->fwd;
    int rc = validate_f32(a, "attn_bwd");
    if (rc != MI_OK) return rc;
    if (!a->o || !a->lse || !b->d_o || !b->dq || !b->dk || !b->dv)
        return mi_fail(MI_E_NULL, "attn_bwd: o, lse, d_o, dq, dk, dv are required");
    if (!mi_aligned16(a->o) || !mi_aligned16(b->d_o) || !mi_aligned16(b->dq) || !mi_aligned16(b->dk) || !mi_aligned16(b->dv))
        return mi_fail(MI_E_ALIGN, "attn_bwd: tensors must be 16-byte aligned");
    if (a->o_stride_token % 4 || a->o_stride_head % 4 || b->dk_stride_token % 4 || b->dk_stride_head % 4 ||
        b->dv_stride_token % 4 || b->dv_stride_head % 4)
        return mi_fail(MI_E_ALIGN, "attn_bwd: strides must be multiples of 4 elements");
    if (a->total_q == 0) return MI_OK;
    const size_t need = (size_t)a->total_q * (size_t)a->n_q_heads * sizeof(float);
    if (!b->workspace || b->workspace_bytes < need || !mi_aligned16(b->workspace))
        return mi_fail(MI_E_WORKSPACE, "attn_bwd: workspace needs %zu bytes (16-byte aligned), got %zu", need, b->workspace_bytes);
    if ((((int64_t)a->total_q + 31) / 32) * a->n_q_heads > 0x7fffffffLL) return mi_fail(MI_E_SHAPE, "attn_bwd: too many work items");
    F32Params fp;
    fill(a, &fp);
    fp.d_o = (const float*)b->d_o; fp.dq = (float*)b->dq; fp.dk = (float*)b->dk; fp.dv = (float*)b->dv;
    fp.m.dk_st = b->dk_stride_token; fp.m.dk_sh = b->dk_stride_head;
    fp.m.dv_st = b->dv_stride_token; fp.m.dv_sh = b->dv_stride_head;
    fp.delta = (float*)b->workspace;
    mi_set_head_split(a, b, &fp.m);
    const size_t kept = mi_attn_bwd_workspace_bytes_f32(a), base = mi_attn_bwd_workspace_bytes_kv(a->total_q, a->total_k, a->n_q_heads, a->n_kv_heads, a->head_dim);
    if (kept > 0 && b->workspace_bytes >= kept) {
        fp.ds = (float*)((char*)b->workspace + (base + 255) / 256 * 256);
        fp.kv_count = ds_heads(a);
        fp.ds_triangle = ds_triangle(a);
    }
    hipStream_t st = (hipStream_t)a->stream;
    switch (a->head_dim) {
        case 32: return launch_bwd_f32<32>(fp, a->flags, st);
        case 64: return launch_bwd_f32<64>(fp, a->flags, st);
        case 96: return launch_bwd_f32<96>(fp, a->flags, st);
        case 128: return launch_bwd_f32<128>(fp, a->flags, st);
        default: return mi_fail(MI_E_SHAPE, "attn_bwd: head_dim %d unsupported", a->head_dim);
    }
}
