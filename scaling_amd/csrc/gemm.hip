// Matrix products of small problems for gfx950: the projections of layers whose products do not fill the chip (and whose
// library calls cost the host more than the device), in every dtype of the package, with the epilogues the layer needs.
//
//     C[m][n] = sum_s sum_k P_s[m][k] Q_s[n][k]  (+ bias[n])  (+ add[m][n])
//
// Each operand is stored either with the contraction index contiguous ("rows": the activations and weights of a forward
// product) or with the contraction index outermost ("kmajor": P[k][m]; the weights of an input gradient, both operands of a
// weight gradient).  Up to three segments s are summed in one pass (the input gradient of projections that share their
// input), and several problems go out in one launch (those projections themselves, or input and weight gradient of one).
//
// What bounds these calls is latency: a 256 x 256 x 256 product is 0.03 GFLOP, and with tiles of 64 x 64 it would keep 16
// compute units busy for four dependent steps.  A workgroup of four wavefronts (2 x 2) therefore owns a TILE x TILE block with
// TILE = 32 until there are enough 64 x 64 blocks to fill the chip; tiles pass global -> registers -> LDS with the loads of the next
// step in flight during the products of the current one, double-buffered, one barrier per step.
//   16-bit: v_mfma_f32_16x16x32 / 32x32x16, kmajor operands through LDS transpose reads
//   fp32:   v_mfma_f32_16x16x4 / 32x32x2, one 128-bit read of a "rows" operand feeds four products (the contraction index is
//           visited in an order in which a lane's four values are consecutive)
#include "common.h"
#include "gemm_wide.h"

#include <type_traits>

int mi_compute_units();

namespace {

typedef float f32x4v __attribute__((ext_vector_type(4)));
typedef short v4i16_t __attribute__((ext_vector_type(4)));
typedef short v8i16_t __attribute__((ext_vector_type(8)));

constexpr int kThreads = 256;
constexpr int kMaxProblems = MI_GEMM_MAX_PROBLEMS, kMaxSegments = MI_GEMM_MAX_SEGMENTS;

struct Segment { const void* p; const void* q; int64_t ldp, ldq; int k; };
struct Problem {
    Segment seg[kMaxSegments];
    void* c; const void* bias; const void* add; void* p_sum;
    int64_t ldc, ldadd;
    int n_seg, p_kmajor, q_kmajor, m, n, tiles_n, first_tile;
};
struct Problems { Problem p[kMaxProblems]; int count; };

template <typename T> struct Mfma;
#define MI_GEMM_MFMA16(T, V8, B16, B32)                                                                                          \
    template <> struct Mfma<T> {                                                                                                 \
        typedef V8 frag_t;                                                                                                       \
        static constexpr int kStep16 = 32, kStep32 = 16;   /* contraction indices per product of the 16- / 32-row shape */       \
        static __device__ __forceinline__ f32x4v mma(frag_t a, frag_t b, f32x4v c) { return B16(a, b, c, 0, 0, 0); }             \
        static __device__ __forceinline__ f32x16_t mma(frag_t a, frag_t b, f32x16_t c) { return B32(a, b, c, 0, 0, 0); }         \
    };
MI_GEMM_MFMA16(__bf16, bf16x8_t, __builtin_amdgcn_mfma_f32_16x16x32_bf16, __builtin_amdgcn_mfma_f32_32x32x16_bf16)
MI_GEMM_MFMA16(_Float16, f16x8_t, __builtin_amdgcn_mfma_f32_16x16x32_f16, __builtin_amdgcn_mfma_f32_32x32x16_f16)
#undef MI_GEMM_MFMA16
template <> struct Mfma<float> {
    typedef f32x4_t frag_t;                                // four products' worth of one lane
    static constexpr int kStep16 = 16, kStep32 = 8;
    static __device__ __forceinline__ f32x4v mma(frag_t a, frag_t b, f32x4v c) {
#pragma unroll
        for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], c, 0, 0, 0);
        return c;
    }
    static __device__ __forceinline__ f32x16_t mma(frag_t a, frag_t b, f32x16_t c) {
#pragma unroll
        for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[i], c, 0, 0, 0);
        return c;
    }
};

// One operand's TILE x BK block in LDS.  BK = 128 (TILE 64) or 256 (TILE 32) bytes of contraction indices.
//   rows:   TILE rows of BK, 16 bytes of padding (16 consecutive rows of a 128-bit read hit all banks once)
//   kmajor: BK rows of TILE elements; the padding puts the rows that one transpose read (16-bit) or the lane groups of one
//           32-bit read (fp32) touch on different banks
template <typename T, int TILE> struct Block {
    static constexpr int kSpan = TILE == 64 ? 128 : 256;
    static constexpr int V = 16 / (int)sizeof(T), BK = kSpan / (int)sizeof(T);
    static constexpr int kRowBytes = kSpan + 16;
    static constexpr int kPad = sizeof(T) == 2 ? (TILE == 64 ? 64 : 0) : (TILE == 64 ? 32 : 16);
    static constexpr int kKBytes = TILE * (int)sizeof(T) + kPad;
    static constexpr int kBytes = TILE * kRowBytes > BK * kKBytes ? TILE * kRowBytes : BK * kKBytes;
    static constexpr int kVecs = TILE * BK / V / kThreads;          // 128-bit vectors per thread
    static_assert(kVecs * kThreads * V == TILE * BK, "whole vectors");

    // vector j of this thread: (row, 16-byte unit) of the block as it is stored in memory
    template <bool KMAJOR> static __device__ __forceinline__ void vec_pos(int j, int& row, int& unit) {
        constexpr int UPR = KMAJOR ? TILE / V : BK / V;
        const int v = (int)threadIdx.x + j * kThreads;
        row = v / UPR;
        unit = v % UPR;
    }
    template <bool KMAJOR> static __device__ __forceinline__ char* vec_addr(char* lds, int j) {
        int row, unit;
        vec_pos<KMAJOR>(j, row, unit);
        return lds + row * (KMAJOR ? kKBytes : kRowBytes) + 16 * unit;
    }
    // Requests the block of rows row0.. and contraction indices k0.. .  Elements outside the matrix are marked in `ok` and
    // zeroed where they are used: their load goes to the first vector of the matrix, so that every load is unconditional and
    // the compiler can count the ones in flight.
    template <bool KMAJOR> static __device__ __forceinline__ void fetch(u32x4_t (&v)[kVecs], bool (&ok)[kVecs], const T* base, int64_t ld, int row0,
                                                                        int rows, int k0, int k) {
#pragma unroll
        for (int j = 0; j < kVecs; ++j) {
            int r, u;
            vec_pos<KMAJOR>(j, r, u);
            const int outer = (KMAJOR ? k0 : row0) + r, inner = (KMAJOR ? row0 : k0) + u * V;
            ok[j] = outer < (KMAJOR ? k : rows) && inner < (KMAJOR ? rows : k);
            const int64_t off = ok[j] ? (int64_t)outer * ld + inner : 0;
            v[j] = *reinterpret_cast<const u32x4_t*>(base + off);
        }
    }
    // fragment of the SHAPE rows from `row` on for the product that covers contraction indices [k, k + step)
    template <bool KMAJOR, int SHAPE> static __device__ __forceinline__ typename Mfma<T>::frag_t frag(const char* lds, int row, int k, int lane) {
        using F = typename Mfma<T>::frag_t;
        const int l = lane % SHAPE, g = lane / SHAPE;      // row of the fragment, group of contraction indices
        if constexpr (!KMAJOR) {
            return *reinterpret_cast<const F*>(lds + (row + l) * kRowBytes + (k + V * g) * (int)sizeof(T));
        } else if constexpr (sizeof(T) == 2) {
            // each block of 16 lanes reads four contraction rows of 16 elements and gets them transposed
            const int i = lane & 15, blk = (lane >> 4) & 1;
            const int col = row + (SHAPE == 32 ? 16 * blk : 0) + 4 * (i & 3);
            const char* a = lds + (k + 8 * g + (i >> 2)) * kKBytes + 2 * col;
            typedef __attribute__((address_space(3))) v4i16_t lds_v4;
            const v4i16_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)(__attribute__((address_space(3))) void*)(void*)a);
            const v4i16_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)(__attribute__((address_space(3))) void*)(void*)(a + 4 * kKBytes));
            return __builtin_bit_cast(F, (v8i16_t)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        } else {
            F x;
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = *reinterpret_cast<const float*>(lds + (k + 4 * g + i) * kKBytes + 4 * (row + l));
            return x;
        }
    }
};

template <typename T, int TILE, bool PK, bool QK>
__device__ __forceinline__ void gemm_tile(const Problem& pr, int tm, int tn, char* smem) {
    using B = Block<T, TILE>;
    constexpr int SHAPE = TILE / 2, STEP = SHAPE == 32 ? Mfma<T>::kStep32 : Mfma<T>::kStep16;
    constexpr int NR = SHAPE * SHAPE / 64;               // accumulator registers
    typedef float acc_t __attribute__((ext_vector_type(NR)));
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = (wave & 1) * SHAPE, wn = (wave >> 1) * SHAPE;
    const int m0 = tm * TILE, n0 = tn * TILE;
    acc_t acc;
#pragma unroll
    for (int r = 0; r < NR; ++r) acc[r] = 0.f;
    float psum[B::V];
#pragma unroll
    for (int i = 0; i < B::V; ++i) psum[i] = 0.f;
    const bool want_sum = PK && pr.p_sum != nullptr && tn == 0;

    // DEPTH steps are in flight: their vectors wait in registers, so a step costs its LDS traffic and a barrier, not a trip
    // to memory (one step ahead, a 3 x 1024 x 1024 product took 8.1 us, 0.5 us per step of 64; now 6.5)
    constexpr int DEPTH = TILE == 64 ? 2 : 4;
    u32x4_t pv[DEPTH][B::kVecs], qv[DEPTH][B::kVecs];
    bool pok[DEPTH][B::kVecs], qok[DEPTH][B::kVecs];
    int seg = 0, k0 = 0, steps = 0;
    for (int i = 0; i < pr.n_seg; ++i) steps += (pr.seg[i].k + B::BK - 1) / B::BK;
    auto fetch = [&](int d) {                              // the next step; past the last one everything is outside the matrix
        const Segment& s = pr.seg[seg];
        B::template fetch<PK>(pv[d], pok[d], (const T*)s.p, s.ldp, m0, pr.m, k0, s.k);
        B::template fetch<QK>(qv[d], qok[d], (const T*)s.q, s.ldq, n0, pr.n, k0, s.k);
        k0 += B::BK;
        if (k0 >= s.k && seg + 1 < pr.n_seg) { k0 = 0; ++seg; }
    };
    auto step = [&](auto d_c) {
        constexpr int d = decltype(d_c)::value;
        char* p_lds = smem + (d & 1) * 2 * B::kBytes;
        char* q_lds = p_lds + B::kBytes;
        const u32x4_t zero = {0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < B::kVecs; ++j) {
            const u32x4_t a = pok[d][j] ? pv[d][j] : zero, b = qok[d][j] ? qv[d][j] : zero;
            if constexpr (PK) {
                if (want_sum) {
                    float f[B::V];
                    Elem<T>::unpack(make_uint4(a[0], a[1], a[2], a[3]), f);
#pragma unroll
                    for (int i = 0; i < B::V; ++i) psum[i] += f[i];
                }
            }
            *reinterpret_cast<u32x4_t*>(B::template vec_addr<PK>(p_lds, j)) = a;
            *reinterpret_cast<u32x4_t*>(B::template vec_addr<QK>(q_lds, j)) = b;
        }
        fetch(d);
        __syncthreads();                                   // this step's blocks are in LDS; the other buffer's readers are done
#pragma unroll
        for (int k = 0; k < B::BK; k += STEP) {
            // A = Q rows (output features), B = P rows: a lane's registers are consecutive features of one output row
            const auto a = B::template frag<QK, SHAPE>(q_lds, wn, k, lane);
            const auto b = B::template frag<PK, SHAPE>(p_lds, wm, k, lane);
            acc = Mfma<T>::mma(a, b, acc);
        }
    };
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) fetch(d);
    for (int i = 0; i < steps; i += DEPTH) {
        step(std::integral_constant<int, 0>{});
        if (i + 1 < steps) step(std::integral_constant<int, 1>{});
        if constexpr (DEPTH == 4) {
            if (i + 2 < steps) step(std::integral_constant<int, 2>{});
            if (i + 3 < steps) step(std::integral_constant<int, 3>{});
        }
    }
    // ---- epilogue: lane = output row, registers in groups of four consecutive features
    const int m = m0 + wm + lane % SHAPE, g = lane / SHAPE;
    if (m < pr.m) {
#pragma unroll
        for (int q = 0; q < NR / 4; ++q) {
            const int n = n0 + wn + (SHAPE == 32 ? 8 * q + 4 * g : 4 * g);
            if (n >= pr.n) continue;                       // n is a multiple of four, as is pr.n
            float x[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = acc[4 * q + i];
            if (pr.bias != nullptr) {
#pragma unroll
                for (int i = 0; i < 4; ++i) x[i] += Elem<T>::load1((const T*)pr.bias + n + i);
            }
            if constexpr (sizeof(T) == 2) {
                typedef T t4 __attribute__((ext_vector_type(4)));
                if (pr.add != nullptr) {
                    // the product is rounded before it is added, as a separate product and sum would round it
                    const t4 a4 = *reinterpret_cast<const t4*>((const T*)pr.add + (int64_t)m * pr.ldadd + n);
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[i] = (float)(T)x[i] + (float)a4[i];
                }
                t4 o;
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = (T)x[i];
                *reinterpret_cast<t4*>((T*)pr.c + (int64_t)m * pr.ldc + n) = o;
            } else {
                if (pr.add != nullptr) {
                    const f32x4_t a4 = *reinterpret_cast<const f32x4_t*>((const float*)pr.add + (int64_t)m * pr.ldadd + n);
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[i] += a4[i];
                }
                const f32x4_t o = {x[0], x[1], x[2], x[3]};
                *reinterpret_cast<f32x4_t*>((float*)pr.c + (int64_t)m * pr.ldc + n) = o;
            }
        }
    }
    if constexpr (PK) {
        if (want_sum) {                                    // the same for the whole workgroup
            // the threads of one 16-byte unit hold the sums of its elements over different contraction rows
            constexpr int UPR = TILE / B::V, ROWS = kThreads / UPR;
            float* lds = reinterpret_cast<float*>(smem);
            __syncthreads();
#pragma unroll
            for (int i = 0; i < B::V; ++i) lds[(tid / UPR) * (TILE + 1) + (tid % UPR) * B::V + i] = psum[i];
            __syncthreads();
            if (tid < TILE && m0 + tid < pr.m) {
                float s = 0.f;
                for (int r = 0; r < ROWS; ++r) s += lds[r * (TILE + 1) + tid];
                Elem<T>::store1((T*)pr.p_sum + m0 + tid, s);
            }
        }
    }
}

template <typename T, int TILE>
__global__ __launch_bounds__(kThreads) void gemm_kernel(const Problems ps) {
    using B = Block<T, TILE>;
    constexpr int kSum = kThreads / (TILE / B::V) * (TILE + 1) * 4;
    constexpr int kLds = 4 * B::kBytes > kSum ? 4 * B::kBytes : kSum;
    __shared__ __attribute__((aligned(16))) char smem[kLds];
    int i = 0;
    while (i + 1 < ps.count && (int)blockIdx.x >= ps.p[i + 1].first_tile) ++i;
    const Problem& pr = ps.p[i];
    const int t = blockIdx.x - pr.first_tile;
    const int tm = t / pr.tiles_n, tn = t - tm * pr.tiles_n;
    if (pr.p_kmajor) gemm_tile<T, TILE, true, true>(pr, tm, tn, smem);
    else if (pr.q_kmajor) gemm_tile<T, TILE, false, true>(pr, tm, tn, smem);
    else gemm_tile<T, TILE, false, false>(pr, tm, tn, smem);
}

// Forward products of a few rows that share their input are weight reads and go to mi_rows_product (3 x 1024 x 1024 in a decode
// step: 9.2 us here, 6.2 there).
template <typename T> bool few_rows(const mi_gemm_problem* in, int count, mi_rows_args& r) {
    if (sizeof(T) != 2 || count > MI_ROWS_MAX_WEIGHTS) return false;
    r = mi_rows_args{};
    for (int i = 0; i < count; ++i) {
        const mi_gemm_problem& a = in[i];
        const auto &s = a.segments[0], &s0 = in[0].segments[0];
        if (a.n_segments != 1 || a.p_kmajor || a.q_kmajor || a.m < 1 || a.m > MI_ROWS_MAX || a.m != in[0].m || s.p != s0.p || s.ldp != s0.ldp || s.k != s0.k ||
            s.k % 32 != 0)
            return false;
        r.w[i] = s.q; r.ldw[i] = s.ldq; r.bias[i] = a.bias; r.add[i] = a.add; r.ldadd[i] = a.ldadd; r.out[i] = a.c; r.ldo[i] = a.ldc; r.n[i] = a.n;
    }
    r.x = in[0].segments[0].p; r.ldx = in[0].segments[0].ldp; r.k = in[0].segments[0].k; r.rows = in[0].m; r.n_weights = count;
    return true;
}

// Calls of 16-bit types with a product of more than 3 GFLOP take the larger blocks of gemm_wide.hip, and below, of 128 rows and more:
//   * gradients, once there are 64 x 64 blocks of weight and input gradient for every compute unit: a block here walks its contraction (tokens; output
//     features) at half the speed.  us, here and there, input and weight gradient of rows x in -> out: 2048 x 768 -> 768 22.7 / 15.7, 512 x 1024 -> 1024 11.5 / 9.7,
//     1024 x 1024 -> 512 12.2 / 9.9, 4096 x 256 -> 256 34 / 18; with fewer blocks level or slower (2048 x 256 -> 512 13.0 / 14.7, 512 x 512 -> 1024 9.0 / 9.4), and with
//     nothing but short contractions (256 x 2048 -> 256 5.7 / 6.2).  Of 212 pairs of 0.1 - 3 GFLOP the rule takes 131, 1.03 - 3.2 x, mean 1.36, and one of .95;
//   * forward products from 1.6 GFLOP on that give three quarters of the compute units such a block: 2048 x 768 -> 768 10.2 / 8.6, 1024 x 1024 -> 1024 10.3 / 9.6, 512 x 768 -> 2048
//     8.7 / 8.4 (below: 512 x 1024 -> 1024 7.8 / 9.4; few long chains: 1024 x 2048 -> 512 13.3 / 14.9);
//   * one forward product over 4096 and more with room to split it: 512 x 4096 -> 512 17.9 / 15.4, 256 x 4096 -> 256 16.6 / 12.4.
// Only whole extents there, as the kernels of this file take them.  What follows a ragged extent inside its last vector meets zeros there (rows of Q past the
// contraction) or unstored results (`ragged`: the entry point allows it); rows must not overlap and a step of them has to be addressable in 31 bits.
bool wide(const mi_gemm_problem* in, int count, int dtype, bool ragged, bool can_split) {
    if (dtype != MI_BF16 && dtype != MI_F16) return false;
    bool large = false, plain = true, forward = true, weights = false, long_chain = can_split && count == 1;     // plain: at least 128 rows, whole extents
    double work = 0;
    int longest = 0;
    int64_t blocks = 0;                                    // of 64 x 64
    for (int i = 0; i < count; ++i) {
        const mi_gemm_problem& a = in[i];
        if (a.m < 0 || a.n <= 0 || a.n_segments < 1 || a.n_segments > kMaxSegments || !a.c || !mi_aligned16(a.c) || a.ldc % 8 ||
            (a.add && (!mi_aligned16(a.add) || a.ldadd % 8)) || (a.p_kmajor && !a.q_kmajor) || (a.p_sum && (!a.p_kmajor || a.n_segments > 1 || a.m % 8)))
            return false;
        for (int s = 0; s < a.n_segments; ++s) {
            const auto& g = a.segments[s];
            const int ep = a.p_kmajor ? a.m : g.k, eq = a.q_kmajor ? a.n : g.k;
            if (!g.p || !g.q || g.k <= 0 || !mi_aligned16(g.p) || !mi_aligned16(g.q) || g.ldp % 8 || g.ldq % 8 || g.ldp < (ep + 7LL) / 8 * 8 ||
                g.ldq < (eq + 7LL) / 8 * 8 || g.ldp >= (1 << 22) || g.ldq >= (1 << 22) || (!a.q_kmajor && g.k % 8) || (!ragged && (a.n % 4 || ep % 8 || eq % 8)))
                return false;
            const double part = 2.0 * a.m * (double)a.n * g.k;
            large = large || part > 3e9;
            work += part;
            longest = std::max(longest, g.k);
            plain = plain && a.n % 4 == 0 && ep % 8 == 0 && eq % 8 == 0;
        }
        plain = plain && (a.p_kmajor ? a.segments[0].k : a.m) >= 128;
        forward = forward && !a.q_kmajor;
        weights = weights || a.p_kmajor;
        long_chain = long_chain && a.n_segments == 1 && a.segments[0].k >= 4096;
        blocks += (int64_t)((a.m + 63) / 64) * ((a.n + 63) / 64);
    }
    if (large || !plain) return large;
    const int64_t units = mi_compute_units();
    return weights ? blocks >= units && longest >= 512 : (work >= 1.6e9 && 4 * blocks >= 3 * units) || (forward && long_chain);
}

int launch_wide(const mi_gemm_problem* in, int count, int dtype, void* workspace, size_t workspace_bytes, hipStream_t st) {
    if (workspace == nullptr || !mi_aligned16(workspace)) workspace_bytes = 0;
    const MiGemmPlan plan = mi_gemm_wide_plan(in, count, workspace_bytes, mi_compute_units());
    return mi_gemm_wide(in, count, dtype, plan, workspace, mi_compute_units(), st);
}

// Without a workspace no contraction is split, and large blocks on a quarter of the chip walk it in one chain: the small ones (or mi_rows_product) keep
// what leaves them less than that or fits one round of 32 x 32.  us, small and large: 64 x 14336 -> 4096 (32 large blocks) 52 / 82, 127 x 4096 -> 4096 (32)
// 21 / 28, 32 x 8192 -> 8192 (64, one round) 37 / 50, 96 x 8192 -> 8192 (64) 64 / 50, 64 x 4096 -> 14336 (112) 53 / 29, 16 x 4096 -> 128256 244 / 181.
bool few_blocks(const mi_gemm_problem* in, int count) {
    int64_t large = 0, small = 0;
    for (int i = 0; i < count; ++i) {
        large += (int64_t)((in[i].m + 127) / 128) * ((in[i].n + 127) / 128);
        small += (int64_t)((in[i].m + 31) / 32) * ((in[i].n + 31) / 32);
    }
    return 4 * large < mi_compute_units() || small <= mi_compute_units();
}

template <typename T> int launch(const mi_gemm_problem* in, int count, hipStream_t st) {
    constexpr int V = Elem<T>::kVec;
    Problems ps;
    ps.count = count;
    int64_t tiles64 = 0;
    for (int i = 0; i < count; ++i) {
        const mi_gemm_problem& a = in[i];
        if (a.m < 0 || a.n <= 0 || a.n % 4 || a.n_segments < 1 || a.n_segments > kMaxSegments)
            return mi_fail(MI_E_SHAPE, "gemm: bad shape m=%d n=%d segments=%d", a.m, a.n, a.n_segments);
        if (!a.c || !mi_aligned16(a.c) || a.ldc % 4 || (a.add && (!mi_aligned16(a.add) || a.ldadd % 4)))
            return mi_fail(MI_E_ALIGN, "gemm: c and add must be 16-byte aligned with leading dimensions that are multiples of 4");
        if (a.p_kmajor && !a.q_kmajor) return mi_fail(MI_E_SHAPE, "gemm: a contraction-major P needs a contraction-major Q");
        if (a.p_sum && !a.p_kmajor) return mi_fail(MI_E_SHAPE, "gemm: p_sum needs a contraction-major P");
        Problem& p = ps.p[i];
        for (int s = 0; s < a.n_segments; ++s) {
            const auto& g = a.segments[s];
            if (!g.p || !g.q || g.k <= 0) return mi_fail(MI_E_NULL, "gemm: empty segment");
            if (!mi_aligned16(g.p) || !mi_aligned16(g.q) || g.ldp % V || g.ldq % V)
                return mi_fail(MI_E_ALIGN, "gemm: operands must be 16-byte aligned with leading dimensions that are multiples of %d", V);
            // the contiguous extent of each operand is read in whole vectors
            if ((a.p_kmajor ? a.m : g.k) % V || (a.q_kmajor ? a.n : g.k) % V)
                return mi_fail(MI_E_SHAPE, "gemm: contiguous extents must be multiples of %d elements", V);
            p.seg[s] = Segment{g.p, g.q, g.ldp, g.ldq, g.k};
        }
        p.c = a.c; p.bias = a.bias; p.add = a.add; p.p_sum = a.p_sum;
        p.ldc = a.ldc; p.ldadd = a.ldadd; p.n_seg = a.n_segments; p.p_kmajor = a.p_kmajor; p.q_kmajor = a.q_kmajor; p.m = a.m; p.n = a.n;
        tiles64 += (int64_t)((a.m + 63) / 64) * ((a.n + 63) / 64);
    }
    // 64 x 64 blocks need half the traffic per product; below one of them per compute unit the finer blocks win on latency
    const int tile = tiles64 >= mi_compute_units() ? 64 : 32;
    int64_t total = 0;
    for (int i = 0; i < count; ++i) {
        Problem& p = ps.p[i];
        p.tiles_n = (p.n + tile - 1) / tile;
        p.first_tile = (int)total;
        total += (int64_t)((p.m + tile - 1) / tile) * p.tiles_n;
        if (total > 0x7fffffffLL) return mi_fail(MI_E_SHAPE, "gemm: too many tiles");
    }
    if (total == 0) return MI_OK;
    mi_rows_args rows;
    if (few_rows<T>(in, count, rows)) {                    // everything has been checked above
        rows.dtype = std::is_same<T, __bf16>::value ? MI_BF16 : MI_F16;
        rows.stream = st;
        return mi_rows_product(&rows);
    }
    if (tile == 64) gemm_kernel<T, 64><<<dim3((unsigned)total), dim3(kThreads), 0, st>>>(ps);
    else gemm_kernel<T, 32><<<dim3((unsigned)total), dim3(kThreads), 0, st>>>(ps);
    return mi_check_launch("gemm");
}

// Column sums of a row-major matrix in fp32 (the bias gradient of a projection whose weight gradient runs on the library):
// a workgroup owns 128 bytes of columns, its 64 groups of 8 lanes walk the rows with eight loads in flight each.  One launch,
// no partial results in memory: 4084 x 3072 bf16 in 11 us (the library sum with its
// semaphore fill 24).
constexpr int kSumThreads = 512, kSumLanes = 8, kSumDepth = 8;

template <typename T>
__global__ __launch_bounds__(kSumThreads) void column_sum_kernel(const T* __restrict__ x, int64_t ld, int rows, int cols, T* __restrict__ out) {
    constexpr int V = Elem<T>::kVec, GROUPS = kSumThreads / kSumLanes, COLS = kSumLanes * V;
    __shared__ float part[GROUPS / 8][COLS + 1];
    const int u = threadIdx.x % kSumLanes, g = threadIdx.x / kSumLanes;
    const int col = blockIdx.x * COLS + u * V;
    const bool live = col < cols;                          // a multiple of V
    float acc[V];
#pragma unroll
    for (int i = 0; i < V; ++i) acc[i] = 0.f;
    const T* base = x + (live ? col : 0);
    auto add = [&](const uint4& v) {
        float f[V];
        Elem<T>::unpack(v, f);
#pragma unroll
        for (int i = 0; i < V; ++i) acc[i] += f[i];
    };
    int r = g;
    for (; r + (kSumDepth - 1) * GROUPS < rows; r += kSumDepth * GROUPS) {
        uint4 v[kSumDepth];
#pragma unroll
        for (int d = 0; d < kSumDepth; ++d) v[d] = *reinterpret_cast<const uint4*>(base + (int64_t)(r + d * GROUPS) * ld);
#pragma unroll
        for (int d = 0; d < kSumDepth; ++d) add(v[d]);
    }
    for (; r < rows; r += GROUPS) add(*reinterpret_cast<const uint4*>(base + (int64_t)r * ld));
    // the eight groups of a wavefront, then the wavefronts, in a fixed order
#pragma unroll
    for (int i = 0; i < V; ++i) {
        acc[i] += __shfl_xor(acc[i], 8, MI_WAVE);
        acc[i] += __shfl_xor(acc[i], 16, MI_WAVE);
        acc[i] += __shfl_xor(acc[i], 32, MI_WAVE);
    }
    if ((threadIdx.x & 63) < kSumLanes) {
#pragma unroll
        for (int i = 0; i < V; ++i) part[threadIdx.x >> 6][u * V + i] = acc[i];
    }
    __syncthreads();
    if (threadIdx.x < COLS && (int)(blockIdx.x * COLS + threadIdx.x) < cols) {
        float s = 0.f;
#pragma unroll
        for (int w = 0; w < GROUPS / 8; ++w) s += part[w][threadIdx.x];
        Elem<T>::store1(out + blockIdx.x * COLS + threadIdx.x, s);
    }
}

template <typename T> int launch_column_sum(const void* x, int64_t ld, int64_t rows, int64_t cols, void* out, hipStream_t st) {
    constexpr int V = Elem<T>::kVec;
    if (cols % V || ld % V || !mi_aligned16(x)) return mi_fail(MI_E_ALIGN, "column_sum: columns and stride must be multiples of %d, x 16-byte aligned", V);
    column_sum_kernel<T><<<dim3((unsigned)((cols + kSumLanes * V - 1) / (kSumLanes * V))), dim3(kSumThreads), 0, st>>>((const T*)x, ld, (int)rows,
                                                                                                                       (int)cols, (T*)out);
    return mi_check_launch("column_sum");
}

// Transposed copy of a 16-bit matrix: 64 x 64 tiles through LDS, 128-bit accesses on both sides, one read and one write of memory.  Columns
// of the output past the last row (up to the next multiple of 8) become zero.  LDS rows of 33 words: a column's 2-byte reads
// spread over the banks.
constexpr int kTransTile = 64;

__global__ __launch_bounds__(256) void transpose_kernel(const uint16_t* __restrict__ x, int64_t ld, int rows, int cols, uint16_t* __restrict__ out,
                                                        int64_t ldo) {
    __shared__ uint32_t tile[kTransTile][kTransTile / 2 + 1];
    const int r0 = blockIdx.y * kTransTile, c0 = blockIdx.x * kTransTile;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int v = (int)threadIdx.x + 256 * j, r = v / 8, u = v % 8;
        u32x4_t w = {0, 0, 0, 0};
        if (r0 + r < rows && c0 + 8 * u < cols) w = *reinterpret_cast<const u32x4_t*>(x + (int64_t)(r0 + r) * ld + c0 + 8 * u);
#pragma unroll
        for (int i = 0; i < 4; ++i) tile[r][4 * u + i] = w[i];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int v = (int)threadIdx.x + 256 * j, c = v / 8, u = v % 8;
        if (c0 + c >= cols || r0 + 8 * u >= rows) continue;
        const uint32_t shift = 16u * (c & 1);
        u32x4_t w;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            w[i] = ((tile[8 * u + 2 * i][c / 2] >> shift) & 0xffffu) | ((tile[8 * u + 2 * i + 1][c / 2] >> shift) << 16);
        *reinterpret_cast<u32x4_t*>(out + (int64_t)(c0 + c) * ldo + r0 + 8 * u) = w;
    }
}

}  // namespace

extern "C" int mi_transpose16(const void* x, int64_t row_stride, int64_t n_rows, int64_t n_cols, void* out, int64_t out_stride, void* stream) {
    if (n_rows < 0 || n_cols < 0 || n_rows > 0x7fffffc0LL || n_cols > 0x7fffffc0LL) return mi_fail(MI_E_SHAPE, "transpose16: bad shape");
    if (n_rows == 0 || n_cols == 0) return MI_OK;
    if (!x || !out) return mi_fail(MI_E_NULL, "transpose16: null pointer");
    if (n_cols % 8 || row_stride % 8 || out_stride % 8 || !mi_aligned16(x) || !mi_aligned16(out))
        return mi_fail(MI_E_ALIGN, "transpose16: columns and strides must be multiples of 8, both matrices 16-byte aligned");
    if (row_stride < n_cols || out_stride < (n_rows + 7) / 8 * 8 || (n_rows + kTransTile - 1) / kTransTile > 65535)
        return mi_fail(MI_E_SHAPE, "transpose16: bad shape or stride");
    const dim3 grid((unsigned)((n_cols + kTransTile - 1) / kTransTile), (unsigned)((n_rows + kTransTile - 1) / kTransTile));
    transpose_kernel<<<grid, dim3(256), 0, (hipStream_t)stream>>>((const uint16_t*)x, row_stride, (int)n_rows, (int)n_cols, (uint16_t*)out, out_stride);
    return mi_check_launch("transpose16");
}

extern "C" int mi_column_sum(const void* x, int64_t row_stride, int64_t n_rows, int64_t n_cols, void* out, int dtype, void* stream) {
    if (!x || !out) return mi_fail(MI_E_NULL, "column_sum: null pointer");
    if (n_rows < 0 || n_cols <= 0 || n_rows > 0x7fffffffLL || n_cols > 0x7fffffffLL || row_stride < n_cols)
        return mi_fail(MI_E_SHAPE, "column_sum: bad shape [%lld, %lld]", (long long)n_rows, (long long)n_cols);
    MI_DISPATCH_DTYPE(dtype, return launch_column_sum<T>(x, row_stride, n_rows, n_cols, out, (hipStream_t)stream));
    return MI_OK;
}

extern "C" int mi_gemm_with_workspace(const mi_gemm_problem* problems, int count, int dtype, void* workspace, size_t workspace_bytes, void* stream) {
    if (!problems || count < 1 || count > kMaxProblems) return mi_fail(MI_E_NULL, "gemm: 1 .. %d problems, got %d", kMaxProblems, count);
    if (wide(problems, count, dtype, true, workspace != nullptr && workspace_bytes > 0)) return launch_wide(problems, count, dtype, workspace, workspace_bytes, (hipStream_t)stream);
    MI_DISPATCH_DTYPE(dtype, return launch<T>(problems, count, (hipStream_t)stream));
    return MI_OK;
}

extern "C" int mi_gemm(const mi_gemm_problem* problems, int count, int dtype, void* stream) {
    if (!problems || count < 1 || count > kMaxProblems) return mi_fail(MI_E_NULL, "gemm: 1 .. %d problems, got %d", kMaxProblems, count);
    if (wide(problems, count, dtype, false, false) && !few_blocks(problems, count)) return launch_wide(problems, count, dtype, nullptr, 0, (hipStream_t)stream);
    MI_DISPATCH_DTYPE(dtype, return launch<T>(problems, count, (hipStream_t)stream));
    return MI_OK;
}

extern "C" size_t mi_gemm_workspace_bytes(const mi_gemm_problem* problems, int count, int dtype) {
    if (!problems || count < 1 || count > kMaxProblems || !wide(problems, count, dtype, true, true)) return 0;
    return mi_gemm_wide_plan(problems, count, (size_t)1 << 30, mi_compute_units()).workspace_bytes;
}
