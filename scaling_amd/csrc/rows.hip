// Products of a few rows for gfx950: what one decode step of up to 16 sequences does with a weight matrix, with the work around it.
//
//     out[m][n] = sum_k X[m][k] W[n][k]   (+ bias[n])   (+ add[m][n])       X = x, or rms_norm(x) * norm_weight
//     out[m][n] = silu(X W0^T) * (X W1^T)                                    (glu)
//
// The weights are read once and nothing else counts, so the design is about having all of them in flight at once: a workgroup owns
// 16 features (32 where there are plenty), its 4 or 8 wavefronts split the contraction, and each requests its share of the weight
// rows from global memory straight in operand layout, eight products ahead.  v_mfma 16x16x32 takes the weights as A and the
// (up to 16) rows as B; the partial sums meet in LDS.  The rows are small enough to be read by every workgroup, so the norm in front
// needs no launch: each wavefront sums the squares of its share of a row, and normalises the operand while it loads it again.
// Up to three matrices that share their input go out in one launch.
//
// What is left is latency: descriptors, then weights and rows, then the norm's barrier, then the sums.  In a decode step of a 4-layer model
// of hidden 1024 (3 sequences) a product of the tiled kernel took 9.2 us, with 3 us for each norm and activation beside
// it.  Wide products run at the rate of the weights: 16 x 4096 -> 128256 191 us, 5.5 TB/s.
//
// Few features leave compute units without a workgroup, and the rest wait for what each of them fetches (1024 features: 64 workgroups, of 16 x k
// weights).  So up to 8 (4) rows may be folded: a workgroup owns 8 (4) features, and a wavefront takes two (four) slices of the contraction at
// once.  Of an operand's 16 rows the first 8 (4) are those of one slice, the next those of the next; of the 16 x 16 results the parts on the
// diagonal count.  The slices and the order that their sums meet in are what they are without, so the results are the same to the bit.
#include "common.h"

namespace {

typedef float f32x4v __attribute__((ext_vector_type(4)));

constexpr int kMaxWeights = MI_ROWS_MAX_WEIGHTS, kMaxRows = MI_ROWS_MAX;
constexpr int kStep = 32;              // contraction indices per product
constexpr int kRedStride = 20;         // floats per row of partial sums: 16-byte aligned, spread over the banks

struct Matrix {
    const void *w, *bias, *add;
    void* out;
    int64_t ldw, ldadd, ldo;
    int n, first_tile;
    __device__ __forceinline__ void arrive() { arrived(w, bias, add, out, ldw, ldadd, ldo, n, first_tile); }
};

struct RowsParams {
    const void *x, *norm_weight;
    int64_t ldx;
    int32_t* count_up;
    int n_weights, rows, k;
    float eps;
    Matrix m[kMaxWeights];
};

template <typename T> struct RowsMfma;
template <> struct RowsMfma<__bf16> {
    typedef bf16x8_t frag_t;
    static __device__ __forceinline__ f32x4v mma(frag_t a, frag_t b, f32x4v c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
};
template <> struct RowsMfma<_Float16> {
    typedef f16x8_t frag_t;
    static __device__ __forceinline__ f32x4v mma(frag_t a, frag_t b, f32x4v c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
};

// TILES: blocks of 16 weight rows per workgroup (2 with GLU: the same 16 rows of both matrices)
// FOLD: slices of the contraction per wavefront; up to 16 / FOLD rows, and 16 / FOLD features of a block
template <typename T, int NW, int TILES, bool NORM, bool GLU, int FOLD>
__global__ __launch_bounds__(64 * NW) void rows_kernel(const RowsParams p) {
    static_assert(!GLU || TILES == 2, "two matrices");
    static_assert(FOLD == 1 || GLU || TILES == 1, "a part of a block");
    using F = typename RowsMfma<T>::frag_t;
    constexpr int CH = TILES == 2 ? 4 : 8;                 // products ahead
    constexpr int SLICES = FOLD * NW, ROWS = kMaxRows / FOLD;     // rows of a slice
    constexpr int FEATURES = (GLU ? 16 : 16 * TILES) / FOLD;
    constexpr int RED = FOLD == 1 ? kRedStride : 16 / FOLD + 4;
    __shared__ __attribute__((aligned(16))) float red[TILES][SLICES][ROWS][RED];
    __shared__ float squares[SLICES][ROWS];
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, G = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // All arguments at once: read where they are used they are a chain of scalar loads from three or four cache lines, each a trip to memory
    // on a fresh launch, before the weights are requested and again in front of the results (with the residual and the second chunk requested
    // up front too, a decode step's five launches per layer at 3 x 1024: 25.0 -> 23.6 us).
    const void *x = p.x, *norm_weight = p.norm_weight;
    int64_t ldx = p.ldx;
    int n_weights = p.n_weights, rows = p.rows, k = p.k;
    int32_t* count_up = p.count_up;
    arrived(x, norm_weight, ldx, n_weights, rows, k, count_up);
    Matrix mx = p.m[0], gate = p.m[1];                     // this workgroup's; GLU: both
    {
        Matrix m2 = p.m[2];
        mx.arrive(); gate.arrive(); m2.arrive();
        if constexpr (!GLU) {
            const bool second = n_weights > 1 && (int)blockIdx.x >= gate.first_tile, third = n_weights > 2 && (int)blockIdx.x >= m2.first_tile;
            if (second) mx = gate;
            if (third) mx = m2;
        }
    }
    const int n0 = ((int)blockIdx.x - mx.first_tile) * FEATURES, n = mx.n;

    // this slice's products: an even number, so that it covers whole 128-byte lines
    const int steps = k / kStep;
    const int per = ((steps + SLICES - 1) / SLICES + 1) & ~1;
    const int part = l16 / ROWS, slice = FOLD * wave + part, row = l16 % ROWS;
    const int s0 = min(slice * per, steps), s1 = min(s0 + per, steps), mine = s1 - s0;
    const int count = __builtin_amdgcn_readfirstlane(mine);                // of the first slice: the others have no more
    const int all = __builtin_amdgcn_readlane(mine, 15);                  // of the last

    // rows past the last one and features past n repeat the last: their results are not stored
    const T* xr = reinterpret_cast<const T*>(x) + (int64_t)min(row, rows - 1) * ldx + 8 * G;
    const T* gr = reinterpret_cast<const T*>(norm_weight) + 8 * G;
    const T* wr[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        const Matrix& m = GLU && t == 1 ? gate : mx;
        wr[t] = reinterpret_cast<const T*>(m.w) + (int64_t)min(n0 + (GLU ? 0 : 16 * t) + row, n - 1) * m.ldw + 8 * G;
    }
    // Weights, rows and norm weights of CH products.  No request is conditional, so that all of them are in flight together: those
    // past this slice's last product repeat it and are not used.
    struct Chunk { u32x4_t w[TILES][CH], x[CH], g[NORM ? CH : 1]; };
    auto request = [&](Chunk& c, int i) {
#pragma unroll
        for (int j = 0; j < CH; ++j) {
            const int64_t at = (int64_t)kStep * min(s0 + i + j, s1 - 1);
            c.x[j] = *reinterpret_cast<const u32x4_t*>(xr + at);
            if constexpr (NORM) c.g[j] = *reinterpret_cast<const u32x4_t*>(gr + at);
#pragma unroll
            for (int t = 0; t < TILES; ++t) c.w[t][j] = *reinterpret_cast<const u32x4_t*>(wr[t] + at);
        }
    };
    Chunk ca, cb;
    if (0 < count) request(ca, 0);
    if (CH < count) request(cb, CH);                       // in front of the loop, where it waits for nothing
    const bool counts = count_up != nullptr && blockIdx.x == 0;
    const int32_t length = (counts ? count_up : reinterpret_cast<const int32_t*>(x))[counts ? min(tid, rows - 1) : 0];

    // bias and residual of the results that this thread stores, requested with the weights, clamped like them and without a branch (in its
    // place the first element of x), which would wait for all that is under way
    constexpr int kOut = (FEATURES * ROWS + 64 * NW - 1) / (64 * NW);
    T bias[kOut], add[kOut];
    if constexpr (!GLU) {
#pragma unroll
        for (int i = 0; i < kOut; ++i) {
            const int idx = tid + i * 64 * NW, m = min(idx / FEATURES, rows - 1), f = min(n0 + idx % FEATURES, n - 1);
            bias[i] = reinterpret_cast<const T*>(mx.bias != nullptr ? mx.bias : x)[mx.bias != nullptr ? f : 0];
            add[i] = reinterpret_cast<const T*>(mx.add != nullptr ? mx.add : x)[mx.add != nullptr ? (int64_t)m * mx.ldadd + f : 0];
        }
    }

    float rstd = 1.f;
    if constexpr (NORM) {
        float ss = 0.f;
        const auto add_squares = [&](const u32x4_t& v) {
            float f[8];
            Elem<T>::unpack(make_uint4(v[0], v[1], v[2], v[3]), f);
#pragma unroll
            for (int i = 0; i < 8; ++i) ss += f[i] * f[i];
        };
        if (0 < count) {
#pragma unroll
            for (int j = 0; j < CH; ++j)
                if (j < mine) add_squares(ca.x[j]);
        }
#pragma unroll 8
        for (int i = CH; i < mine; ++i) add_squares(*reinterpret_cast<const u32x4_t*>(xr + kStep * (s0 + i)));
        ss += __shfl_xor(ss, 16, MI_WAVE);
        ss += __shfl_xor(ss, 32, MI_WAVE);
        if (G == 0) squares[slice][row] = ss;
        __syncthreads();
        float total = 0.f;
#pragma unroll
        for (int w = 0; w < SLICES; ++w) total += squares[w][row];
        rstd = rsqrtf(total / (float)k + p.eps);
    }

    f32x4v acc[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t) acc[t] = f32x4v{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const Chunk& c, int i) {
#pragma unroll
        for (int j = 0; j < CH; ++j) {
            uint4 xv = make_uint4(c.x[j][0], c.x[j][1], c.x[j][2], c.x[j][3]);
            if constexpr (NORM) {
                float f[8], g[8];
                Elem<T>::unpack(xv, f);
                Elem<T>::unpack(make_uint4(c.g[j][0], c.g[j][1], c.g[j][2], c.g[j][3]), g);
#pragma unroll
                for (int e = 0; e < 8; ++e) f[e] = (f[e] * rstd) * g[e];
                xv = Elem<T>::pack(f);
            }
            if (i + j < count) {                           // the same for the whole wavefront
                u32x4_t w[TILES];
#pragma unroll
                for (int t = 0; t < TILES; ++t) w[t] = c.w[t][j];
                if (FOLD > 1 && i + j >= all && i + j >= mine) {   // nothing more of this slice
                    xv = make_uint4(0, 0, 0, 0);
#pragma unroll
                    for (int t = 0; t < TILES; ++t) w[t] = u32x4_t{0, 0, 0, 0};
                }
#pragma unroll
                for (int t = 0; t < TILES; ++t) acc[t] = RowsMfma<T>::mma(__builtin_bit_cast(F, w[t]), __builtin_bit_cast(F, xv), acc[t]);
            }
        }
    };
    for (int i = 0; i < count; i += 2 * CH) {
        multiply(ca, i);
        if (i + 2 * CH < count) request(ca, i + 2 * CH);
        if (i + CH < count) {
            multiply(cb, i + CH);
            if (i + 3 * CH < count) request(cb, i + 3 * CH);
        }
    }

    // a lane holds four consecutive features of a row
    if (FOLD == 1 || G * FOLD / 4 == part) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) *reinterpret_cast<f32x4v*>(&red[t][slice][row][4 * (G % (4 / FOLD))]) = acc[t];
    }
    __syncthreads();
    if (counts && tid < rows) count_up[tid] = length + 1;
#pragma unroll
    for (int i = 0; i < kOut; ++i) {
        const int idx = tid + i * 64 * NW, m = idx / FEATURES, f = idx % FEATURES;
        if (m >= rows || n0 + f >= n) continue;
        const auto total = [&](int t, int c) {
            float s = 0.f;
#pragma unroll
            for (int w = 0; w < SLICES; ++w) s += red[t][w][m][c];
            return s;
        };
        T* out = reinterpret_cast<T*>(mx.out) + (int64_t)m * mx.ldo + n0 + f;
        if constexpr (GLU) {
            // both products are rounded as separate launches would store them
            const float a = (float)(T)total(0, f), g = (float)(T)total(1, f);
            *out = (T)((a * (1.0f / (1.0f + __expf(-a)))) * g);
        } else {
            float v = total(f / 16, f % 16);
            if (mx.bias != nullptr) v += (float)bias[i];
            if (mx.add != nullptr) v = (float)(T)v + (float)add[i];
            *out = (T)v;
        }
    }
}

template <typename T, int NW, int TILES, bool GLU, int FOLD> void launch_one(const RowsParams& p, int grid, hipStream_t st) {
    if (p.norm_weight != nullptr) rows_kernel<T, NW, TILES, true, GLU, FOLD><<<dim3((unsigned)grid), dim3(64 * NW), 0, st>>>(p);
    else rows_kernel<T, NW, TILES, false, GLU, FOLD><<<dim3((unsigned)grid), dim3(64 * NW), 0, st>>>(p);
}

template <typename T> int launch(const mi_rows_args& a, hipStream_t st) {
    RowsParams p{};
    p.x = a.x; p.norm_weight = a.norm_weight; p.ldx = a.ldx; p.count_up = a.count_up;
    p.n_weights = a.n_weights; p.rows = a.rows; p.k = a.k; p.eps = a.eps;
    int64_t blocks16 = 0;
    for (int i = 0; i < a.n_weights; ++i) {
        p.m[i] = Matrix{a.w[i], a.bias[i], a.add[i], a.out[i], a.ldw[i], a.ldadd[i], a.ldo[i], a.n[i], 0};
        if (i == 0 || !a.glu) blocks16 += (a.n[i] + 15) / 16;
    }
    // Two blocks per workgroup once that leaves four workgroups per compute unit: the rows are read half as often.  Eight wavefronts
    // while there is less than one workgroup of four per SIMD, to have more of the weights in flight.
    const bool wide = !a.glu && blocks16 >= 2048, many = blocks16 >= 1024;
    // Folded where a compute unit (of 256: the lines count blocks) is left with less: 256 workgroups of a quarter or of half a block instead of as many whole ones or fewer, or three halves on
    // a compute unit instead of two blocks.  us, one / two / four slices, weights from memory: 3 rows, k 1024 -> 1024 4.53 / 3.60 / 3.16, 2816 -> 1024 7.09 / 5.59 /
    // 4.44, 4096 -> 1024 with norm and glu 14.9 / 11.2 / 9.1; 1024 -> 1536 4.77 / 3.90 / 4.20; 4096 -> 6144 15.3 / 13.6 / 14.6 (8 rows 17.2 / 16.3); elsewhere
    // the rows are only read more often: 1024 -> 2816 4.87 / 5.23 / 4.96, 4096 -> 4096 9.00 / 10.0 / 10.7, 8 rows, 4096 -> 10240 25.5 / 27.2.
    const int fold = a.rows <= 4 && blocks16 <= 64 ? 4 : a.rows <= 8 && (blocks16 <= 128 || (blocks16 > 256 && blocks16 <= 384)) ? 2 : 1;
    const int features = (wide ? 32 : 16) / fold;
    int64_t grid = 0;
    for (int i = 0; i < (a.glu ? 1 : a.n_weights); ++i) {
        p.m[i].first_tile = (int)grid;
        grid += (a.n[i] + features - 1) / features;
    }
    if (grid > 0x7fffffffLL) return mi_fail(MI_E_SHAPE, "rows: too many features");
    if (fold == 4) a.glu ? launch_one<T, 2, 2, true, 4>(p, (int)grid, st) : launch_one<T, 2, 1, false, 4>(p, (int)grid, st);
    else if (fold == 2) a.glu ? launch_one<T, 4, 2, true, 2>(p, (int)grid, st) : launch_one<T, 4, 1, false, 2>(p, (int)grid, st);
    else if (a.glu) many ? launch_one<T, 4, 2, true, 1>(p, (int)grid, st) : launch_one<T, 8, 2, true, 1>(p, (int)grid, st);
    else if (wide) launch_one<T, 4, 2, false, 1>(p, (int)grid, st);
    else many ? launch_one<T, 4, 1, false, 1>(p, (int)grid, st) : launch_one<T, 8, 1, false, 1>(p, (int)grid, st);
    return mi_check_launch("rows");
}

}  // namespace

extern "C" int mi_rows_product(const mi_rows_args* a) {
    if (!a || !a->x) return mi_fail(MI_E_NULL, "rows: null pointer");
    if (a->rows < 1 || a->rows > kMaxRows || a->k <= 0 || a->k % kStep || a->n_weights < 1 || a->n_weights > kMaxWeights || (a->glu && a->n_weights != 2))
        return mi_fail(MI_E_SHAPE, "rows: 1 .. %d rows, k a multiple of %d, 1 .. %d weights (2 with glu); got %d, %d, %d", kMaxRows, kStep, kMaxWeights,
                       a->rows, a->k, a->n_weights);
    if (!mi_aligned16(a->x) || a->ldx % 8 || (a->norm_weight && !mi_aligned16(a->norm_weight)))
        return mi_fail(MI_E_ALIGN, "rows: x and norm weight must be 16-byte aligned, the row stride a multiple of 8");
    for (int i = 0; i < a->n_weights; ++i) {
        if (!a->w[i] || (!a->out[i] && !(a->glu && i == 1))) return mi_fail(MI_E_NULL, "rows: null pointer");
        if (a->n[i] <= 0 || (a->glu && a->n[i] != a->n[0]) || a->ldw[i] < a->k) return mi_fail(MI_E_SHAPE, "rows: bad weight shape");
        if (!mi_aligned16(a->w[i]) || a->ldw[i] % 8) return mi_fail(MI_E_ALIGN, "rows: weights must be 16-byte aligned with rows of whole vectors");
    }
    switch (a->dtype) {
        case MI_BF16: return launch<__bf16>(*a, (hipStream_t)a->stream);
        case MI_F16: return launch<_Float16>(*a, (hipStream_t)a->stream);
        default: return mi_fail(MI_E_DTYPE, "rows: bf16 or f16 tensors (dtype code %d)", a->dtype);
    }
}
