// Stand-alone rotary embedding (rotate-half pairing) for gfx950: one pass, 128-bit accesses.
//
// One thread owns a 128-bit vector of the first half of the rotated span and its partner vector
// rot_dim/2 further on, so both outputs of every (i, i + rot_dim/2) pair come from one thread.  The
// features beyond rot_dim are copied.  A scalar kernel covers head sizes that do not vectorise.  q and k, which share tables and
// positions, go in one launch as heads of two tensors: as two they took 4.1 us each for 256 tokens of 4 heads of 64 (float32), 4.3 together.
#include "common.h"

namespace {

constexpr int kBlock = 256;

struct RotaryParams {
    const void* x; void* out; const void* cos; const void* sin; const int64_t* pos;
    int64_t n_tokens; int n_heads; int head_dim; int rot_dim;
    int64_t xs_t, xs_h, os_t, os_h;
    int64_t table_rows, seq_len_null; float sign;
    const void* x2; void* out2; int64_t xs2_t, xs2_h, os2_t, os2_h;        // of a second tensor: heads first .. n_heads - 1
    int first;                                             // n_heads without one
};

// x and out of a head's first feature
template <typename T> __device__ __forceinline__ void head_rows(const RotaryParams& p, int64_t t, int h, const T*& x, T*& out) {
    if (h < p.first) {
        x = (const T*)p.x + t * p.xs_t + (int64_t)h * p.xs_h;
        out = (T*)p.out + t * p.os_t + (int64_t)h * p.os_h;
    } else {
        x = (const T*)p.x2 + t * p.xs2_t + (int64_t)(h - p.first) * p.xs2_h;
        out = (T*)p.out2 + t * p.os2_t + (int64_t)(h - p.first) * p.os2_h;
    }
}

__device__ __forceinline__ int64_t table_row(const RotaryParams& p, int64_t t) {
    int64_t r = p.pos ? p.pos[t] : (t % p.seq_len_null);
    if (r < 0) r = 0;
    if (r >= p.table_rows) r = p.table_rows - 1;
    return r;
}

// reads N consecutive table values (N = 4 or 8) starting at a 16-byte aligned address
template <typename TT, int N> __device__ __forceinline__ void load_table(const TT* ptr, float* f) {
    if constexpr (sizeof(TT) == 4) {
#pragma unroll
        for (int j = 0; j < N / 4; ++j) Elem<float>::unpack(reinterpret_cast<const uint4*>(ptr)[j], f + 4 * j);
    } else {
        static_assert(N == 8, "16-bit tables are read 8 values at a time");
        Elem<TT>::unpack(*reinterpret_cast<const uint4*>(ptr), f);
    }
}

// One vector of either half of a head, rotated: what every kernel here leaves for a data type and 16-bit tables of the same type.
template <typename T>
__device__ __forceinline__ void rotate_half(const float* x0, const float* x1, const float* cA, const float* sA, const float* cB, const float* sB, uint4& lo, uint4& hi) {
    constexpr int V = Elem<T>::kVec;
    float o0[V], o1[V];
    if constexpr (std::is_same_v<T, _Float16>) {           // first half rounded twice, second half once
        uint32_t h[4];
#pragma unroll
        for (int i = 0; i < V; ++i) o0[i] = sum_f32(x0[i], cA[i], -(x1[i] * sA[i]));
#pragma unroll
        for (int i = 0; i < 4; ++i) h[i] = fma_pair_f16(x1[2 * i], cB[2 * i], x0[2 * i] * sB[2 * i], x1[2 * i + 1], cB[2 * i + 1], x0[2 * i + 1] * sB[2 * i + 1]);
        lo = Elem<T>::pack(o0);
        hi = make_uint4(h[0], h[1], h[2], h[3]);
    } else {
#pragma unroll
        for (int i = 0; i < V; ++i) {
            o0[i] = x0[i] * cA[i] - x1[i] * sA[i];
            o1[i] = x1[i] * cB[i] + x0[i] * sB[i];
        }
        lo = Elem<T>::pack(o0);
        hi = Elem<T>::pack(o1);
    }
}

// T: data type, TT: table type.  Work item = (token, head, vec) with vec over half the rotated span
// followed by the vectors of the unrotated tail.
template <typename T, typename TT>
__global__ __launch_bounds__(kBlock) void rotary_vec_kernel(RotaryParams p) {
    constexpr int V = Elem<T>::kVec;
    const int half_vecs = p.rot_dim / 2 / V;
    const int tail_vecs = (p.head_dim - p.rot_dim) / V;
    const int per_head = half_vecs + tail_vecs;
    const int64_t per_token = (int64_t)per_head * p.n_heads;
    const int64_t item = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (item >= per_token * p.n_tokens) return;
    const int64_t t = item / per_token;
    const int rem = (int)(item % per_token);
    const int h = rem / per_head;
    const int v = rem % per_head;
    const T* xrow;
    T* orow;
    head_rows(p, t, h, xrow, orow);
    if (v >= half_vecs) {  // unrotated tail
        const int c = p.rot_dim + (v - half_vecs) * V;
        if ((const void*)xrow != (const void*)orow)
            stg_nt(reinterpret_cast<uint4*>(orow + c), *reinterpret_cast<const uint4*>(xrow + c));
        return;
    }
    const int c0 = v * V, c1 = c0 + p.rot_dim / 2;
    const int64_t r = table_row(p, t);
    const TT* cr = (const TT*)p.cos + r * p.rot_dim;
    const TT* sr = (const TT*)p.sin + r * p.rot_dim;
    float x0[V], x1[V], cA[V], sA[V], cB[V], sB[V];
    Elem<T>::unpack(ldg_nt(reinterpret_cast<const uint4*>(xrow + c0)), x0);
    Elem<T>::unpack(ldg_nt(reinterpret_cast<const uint4*>(xrow + c1)), x1);
    load_table<TT, V>(cr + c0, cA);
    load_table<TT, V>(sr + c0, sA);
    load_table<TT, V>(cr + c1, cB);
    load_table<TT, V>(sr + c1, sB);
    uint4 lo, hi;
    if constexpr (sizeof(TT) == 2) {
#pragma unroll
        for (int i = 0; i < V; ++i) {
            sA[i] *= p.sign;
            sB[i] *= p.sign;
        }
        rotate_half<T>(x0, x1, cA, sA, cB, sB, lo, hi);
    } else {
        float o0[V], o1[V];
#pragma unroll
        for (int i = 0; i < V; ++i) {
            o0[i] = x0[i] * cA[i] - x1[i] * (p.sign * sA[i]);
            o1[i] = x1[i] * cB[i] + x0[i] * (p.sign * sB[i]);
        }
        lo = Elem<T>::pack(o0);
        hi = Elem<T>::pack(o1);
    }
    stg_nt(reinterpret_cast<uint4*>(orow + c0), lo);
    stg_nt(reinterpret_cast<uint4*>(orow + c1), hi);
}

// What a prefill leaves in a KV cache, in one launch: k rotated (whole head, rotate-half or interleaved pairs, as the two kernels around this one)
// into the cache and, packed, for the attention launch that follows; v into the cache; the context lengths.  A thread owns a vector of the
// first half of a k row and its partner (interleaved: one of either half) or the same two of a v row.  As two rotary launches (q and k; bfloat16 q is now
// rotated where the attention kernel loads it), two copies and a fill it was five launches a layer.
struct FillParams {
    const void *k, *v, *cos, *sin;
    const int64_t* pos;
    void *k_out, *k_cache, *v_cache;
    int32_t* ctx_len;
    int64_t n_tokens, k_st, k_sh, v_st, v_sh, c_sb, c_st, c_sh, table_rows;
    int seq, n_heads, batch;
};

template <typename T, int D, bool PAIRS>
__global__ __launch_bounds__(kBlock) void fill_cache_kernel(const FillParams p) {
    constexpr int V = Elem<T>::kVec, HALF = D / 2 / V;
    const uint32_t item = blockIdx.x * (uint32_t)kBlock + threadIdx.x;        // fewer than 2^32: checked by the entry point
    if (item < (uint32_t)p.batch) p.ctx_len[item] = p.seq;
    const uint32_t per_token = 2u * HALF * p.n_heads, token = item / per_token;
    if (token >= (uint32_t)p.n_tokens) return;
    const uint32_t rem = item - token * per_token, b = token / (uint32_t)p.seq;
    const int h = rem / (2 * HALF), c = rem % HALF;
    const bool value = rem % (2 * HALF) >= HALF;
    const int64_t t = token, at = (int64_t)b * p.c_sb + (int64_t)(token - b * p.seq) * p.c_st + (int64_t)h * p.c_sh + V * c;
    const T* src = value ? (const T*)p.v + t * p.v_st + (int64_t)h * p.v_sh + V * c : (const T*)p.k + t * p.k_st + (int64_t)h * p.k_sh + V * c;
    uint4 lo = *reinterpret_cast<const uint4*>(src), hi = *reinterpret_cast<const uint4*>(src + D / 2);
    if (value) {
        T* dst = (T*)p.v_cache + at;
        *reinterpret_cast<uint4*>(dst) = lo;
        *reinterpret_cast<uint4*>(dst + D / 2) = hi;
        return;
    }
    int64_t r = p.pos[t];
    r = r < 0 ? 0 : (r >= p.table_rows ? p.table_rows - 1 : r);
    float x0[V], x1[V];
    Elem<T>::unpack(lo, x0);
    Elem<T>::unpack(hi, x1);
    if constexpr (PAIRS) {
        const float *cr = (const float*)p.cos + r * (D / 2) + V / 2 * c, *sr = (const float*)p.sin + r * (D / 2) + V / 2 * c;
#pragma unroll
        for (int i = 0; i < V / 2; ++i) {
            rotate_complex_pair(x0[2 * i], x0[2 * i + 1], cr[i], sr[i]);
            rotate_complex_pair(x1[2 * i], x1[2 * i + 1], cr[D / 4 + i], sr[D / 4 + i]);
        }
        lo = Elem<T>::pack(x0);
        hi = Elem<T>::pack(x1);
    } else {
        float cA[V], sA[V], cB[V], sB[V];
        load_table<T, V>((const T*)p.cos + r * D + V * c, cA);
        load_table<T, V>((const T*)p.sin + r * D + V * c, sA);
        load_table<T, V>((const T*)p.cos + r * D + D / 2 + V * c, cB);
        load_table<T, V>((const T*)p.sin + r * D + D / 2 + V * c, sB);
        rotate_half<T>(x0, x1, cA, sA, cB, sB, lo, hi);
    }
    T *dst = (T*)p.k_cache + at, *out = (T*)p.k_out + (t * p.n_heads + h) * D + V * c;
    *reinterpret_cast<uint4*>(dst) = lo;
    *reinterpret_cast<uint4*>(dst + D / 2) = hi;
    *reinterpret_cast<uint4*>(out) = lo;
    *reinterpret_cast<uint4*>(out + D / 2) = hi;
}

template <typename T, typename TT>
__global__ __launch_bounds__(kBlock) void rotary_scalar_kernel(RotaryParams p) {
    const int half = p.rot_dim / 2;
    const int per_head = half + (p.head_dim - p.rot_dim);
    const int64_t per_token = (int64_t)per_head * p.n_heads;
    const int64_t item = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (item >= per_token * p.n_tokens) return;
    const int64_t t = item / per_token;
    const int rem = (int)(item % per_token);
    const int h = rem / per_head;
    const int i = rem % per_head;
    const T* xrow;
    T* orow;
    head_rows(p, t, h, xrow, orow);
    if (i >= half) {
        const int c = p.rot_dim + (i - half);
        Elem<T>::store1(orow + c, Elem<T>::load1(xrow + c));
        return;
    }
    const int64_t r = table_row(p, t);
    const TT* cr = (const TT*)p.cos + r * p.rot_dim;
    const TT* sr = (const TT*)p.sin + r * p.rot_dim;
    const float x0 = Elem<T>::load1(xrow + i), x1 = Elem<T>::load1(xrow + i + half);
    const float o0 = x0 * Elem<TT>::load1(cr + i) - x1 * (p.sign * Elem<TT>::load1(sr + i));
    const float o1 = x1 * Elem<TT>::load1(cr + i + half) + x0 * (p.sign * Elem<TT>::load1(sr + i + half));
    Elem<T>::store1(orow + i, o0);
    Elem<T>::store1(orow + i + half, o1);
}

// Interleaved ("complex") pairing (2i, 2i+1) over the whole head, fp32 tables [rows, head_dim/2].
// One thread owns one 128-bit vector = V/2 complete pairs.
template <typename T>
__global__ __launch_bounds__(kBlock) void rotary_complex_kernel(RotaryParams p) {
    constexpr int V = Elem<T>::kVec;
    const int vec_per_head = p.head_dim / V;
    const int64_t per_token = (int64_t)vec_per_head * p.n_heads;
    const int64_t item = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (item >= per_token * p.n_tokens) return;
    const int64_t t = item / per_token;
    const int rem = (int)(item % per_token);
    const int h = rem / vec_per_head, v = rem % vec_per_head;
    const T* xrow;
    T* orow;
    head_rows(p, t, h, xrow, orow);
    xrow += v * V;
    orow += v * V;
    const int64_t r = table_row(p, t);
    const float* cr = (const float*)p.cos + r * (p.head_dim / 2) + v * (V / 2);
    const float* sr = (const float*)p.sin + r * (p.head_dim / 2) + v * (V / 2);
    float x[V], o[V];
    Elem<T>::unpack(*reinterpret_cast<const uint4*>(xrow), x);
#pragma unroll
    for (int i = 0; i < V / 2; ++i) {
        o[2 * i] = x[2 * i];
        o[2 * i + 1] = x[2 * i + 1];
        rotate_complex_pair(o[2 * i], o[2 * i + 1], cr[i], p.sign * sr[i]);
    }
    stg_nt(reinterpret_cast<uint4*>(orow), Elem<T>::pack(o));
}

RotaryParams params(const mi_rotary_rows& r, const void* cos, const void* sin, const int64_t* position_ids, int64_t n_tokens, int32_t head_dim, int32_t rot_dim,
                    int64_t table_rows, int64_t seq_len_for_null_ids, int inverse) {
    return RotaryParams{r.x, r.out, cos, sin, position_ids, n_tokens, r.n_heads, head_dim, rot_dim, r.x_stride_token, r.x_stride_head, r.out_stride_token,
                        r.out_stride_head, table_rows, seq_len_for_null_ids, inverse ? -1.0f : 1.0f, nullptr, nullptr, 0, 0, 0, 0, r.n_heads};
}

// whether rows and heads of both tensors are whole vectors
template <typename T> bool whole(const RotaryParams& p) {
    constexpr int V = Elem<T>::kVec;
    return p.xs_t % V == 0 && p.xs_h % V == 0 && p.os_t % V == 0 && p.os_h % V == 0 && p.xs2_t % V == 0 && p.xs2_h % V == 0 && p.os2_t % V == 0 &&
           p.os2_h % V == 0 && mi_aligned16(p.x) && mi_aligned16(p.out) && mi_aligned16(p.x2) && mi_aligned16(p.out2);
}

template <typename T, typename TT> int launch(const RotaryParams& p, hipStream_t st) {
    constexpr int V = Elem<T>::kVec;
    const bool vec_ok = (p.rot_dim / 2) % V == 0 && (p.head_dim - p.rot_dim) % V == 0 && whole<T>(p) &&
                        mi_aligned16(p.cos) && mi_aligned16(p.sin) && (sizeof(TT) == 4 || V == 8);
    int64_t per_head = vec_ok ? (p.rot_dim / 2 / V + (p.head_dim - p.rot_dim) / V) : (p.rot_dim / 2 + p.head_dim - p.rot_dim);
    const int64_t items = per_head * p.n_heads * p.n_tokens;
    const int64_t blocks = (items + kBlock - 1) / kBlock;
    if (blocks > 0x7fffffffLL) return mi_fail(MI_E_SHAPE, "rotary: too many elements");
    if (vec_ok)
        rotary_vec_kernel<T, TT><<<dim3((unsigned)blocks), dim3(kBlock), 0, st>>>(p);
    else
        rotary_scalar_kernel<T, TT><<<dim3((unsigned)blocks), dim3(kBlock), 0, st>>>(p);
    return mi_check_launch("rotary");
}

int rotate(const RotaryParams& p, int dtype, int table_dtype, hipStream_t st) {
    if (!p.x || !p.out || !p.cos || !p.sin) return mi_fail(MI_E_NULL, "rotary: null pointer");
    if (p.n_tokens < 0 || p.n_heads <= 0 || p.head_dim <= 0 || p.rot_dim <= 1 || p.rot_dim > p.head_dim || (p.rot_dim & 1) || p.table_rows <= 0)
        return mi_fail(MI_E_SHAPE, "rotary: bad shape tokens=%lld heads=%d head_dim=%d rot_dim=%d table_rows=%lld",
                       (long long)p.n_tokens, p.n_heads, p.head_dim, p.rot_dim, (long long)p.table_rows);
    if (!p.pos && p.seq_len_null <= 0) return mi_fail(MI_E_SHAPE, "rotary: need position ids or a sequence length");
    if (table_dtype != dtype && table_dtype != MI_F32) return mi_fail(MI_E_DTYPE, "rotary: table dtype must equal the data dtype or be fp32");
    MI_DISPATCH_DTYPE(dtype, {
        if (table_dtype == dtype) return launch<T, T>(p, st);
        return launch<T, float>(p, st);
    });
    return MI_OK;
}

int rotate_complex(const RotaryParams& p, int dtype, hipStream_t st) {
    if (!p.x || !p.out || !p.cos || !p.sin) return mi_fail(MI_E_NULL, "rotary_complex: null pointer");
    if (p.n_tokens < 0 || p.n_heads <= 0 || p.head_dim <= 0 || p.table_rows <= 0)
        return mi_fail(MI_E_SHAPE, "rotary_complex: bad shape tokens=%lld heads=%d head_dim=%d", (long long)p.n_tokens, p.n_heads, p.head_dim);
    if (!p.pos && p.seq_len_null <= 0) return mi_fail(MI_E_SHAPE, "rotary_complex: need position ids or a sequence length");
    MI_DISPATCH_DTYPE(dtype, {
        constexpr int V = Elem<T>::kVec;
        if (p.head_dim % V || !whole<T>(p))
            return mi_fail(MI_E_ALIGN, "rotary_complex: head_dim and strides must be multiples of %d elements, pointers 16-byte aligned", V);
        const int64_t items = (int64_t)(p.head_dim / V) * p.n_heads * p.n_tokens;
        const int64_t blocks = (items + kBlock - 1) / kBlock;
        if (blocks > 0x7fffffffLL) return mi_fail(MI_E_SHAPE, "rotary_complex: too many elements");
        rotary_complex_kernel<T><<<dim3((unsigned)blocks), dim3(kBlock), 0, st>>>(p);
    });
    return mi_check_launch("rotary_complex");
}

}  // namespace

extern "C" int mi_rotary(const void* x, void* out, const void* cos, const void* sin, const int64_t* position_ids,
                         int64_t n_tokens, int32_t n_heads, int32_t head_dim, int32_t rot_dim, int64_t x_stride_token,
                         int64_t x_stride_head, int64_t out_stride_token, int64_t out_stride_head, int64_t table_rows,
                         int64_t seq_len_for_null_ids, int inverse, int dtype, int table_dtype, void* stream) {
    if (n_tokens == 0) return MI_OK;       // nothing to do (an empty tensor may come with a null pointer)
    const mi_rotary_rows r{x, out, x_stride_token, x_stride_head, out_stride_token, out_stride_head, n_heads};
    return rotate(params(r, cos, sin, position_ids, n_tokens, head_dim, rot_dim, table_rows, seq_len_for_null_ids, inverse), dtype, table_dtype,
                  (hipStream_t)stream);
}

extern "C" int mi_rotary_complex(const void* x, void* out, const float* cos, const float* sin, const int64_t* position_ids,
                                 int64_t n_tokens, int32_t n_heads, int32_t head_dim, int64_t x_stride_token,
                                 int64_t x_stride_head, int64_t out_stride_token, int64_t out_stride_head,
                                 int64_t table_rows, int64_t seq_len_for_null_ids, int inverse, int dtype, void* stream) {
    if (n_tokens == 0) return MI_OK;       // nothing to do (an empty tensor may come with a null pointer)
    const mi_rotary_rows r{x, out, x_stride_token, x_stride_head, out_stride_token, out_stride_head, n_heads};
    return rotate_complex(params(r, cos, sin, position_ids, n_tokens, head_dim, head_dim, table_rows, seq_len_for_null_ids, inverse), dtype, (hipStream_t)stream);
}

// One launch where each tensor alone would take the kernel that both together take; else one after the other.
extern "C" int mi_rotary_two(const mi_rotary_rows* rows, const void* cos, const void* sin, const int64_t* position_ids, int64_t n_tokens, int32_t head_dim,
                             int32_t rot_dim, int64_t table_rows, int64_t seq_len_for_null_ids, int inverse, int interleaved, int dtype, int table_dtype,
                             void* stream) {
    if (n_tokens == 0) return MI_OK;
    if (!rows || !rows[1].x || !rows[1].out) return mi_fail(MI_E_NULL, "rotary: null pointer");
    if (rows[0].n_heads <= 0 || rows[1].n_heads <= 0 || (interleaved && (rot_dim != head_dim || table_dtype != MI_F32)))
        return mi_fail(MI_E_SHAPE, "rotary: heads %d and %d; interleaved pairs cover the head, with fp32 tables", rows[0].n_heads, rows[1].n_heads);
    const auto one = [&](const RotaryParams& p) { return interleaved ? rotate_complex(p, dtype, (hipStream_t)stream) : rotate(p, dtype, table_dtype, (hipStream_t)stream); };
    RotaryParams p = params(rows[0], cos, sin, position_ids, n_tokens, head_dim, rot_dim, table_rows, seq_len_for_null_ids, inverse);
    const RotaryParams second = params(rows[1], cos, sin, position_ids, n_tokens, head_dim, rot_dim, table_rows, seq_len_for_null_ids, inverse);
    const bool f32 = dtype == MI_F32;                      // vectors of 4 elements, of 8 for both 16-bit types
    const auto fits = [&](const RotaryParams& r) { return f32 ? whole<float>(r) : whole<_Float16>(r); };
    if (fits(p) && fits(second) && rows[0].n_heads <= 0x7fffffff - rows[1].n_heads) {
        p.n_heads += second.n_heads;
        p.x2 = second.x; p.out2 = second.out; p.xs2_t = second.xs_t; p.xs2_h = second.xs_h; p.os2_t = second.os_t; p.os2_h = second.os_h;
        return one(p);
    }
    if (const int rc = one(p); rc != MI_OK) return rc;
    return one(second);
}

extern "C" int mi_fill_cache(const mi_fill_cache_args* a) {
    if (!a) return mi_fail(MI_E_NULL, "fill_cache: args is null");
    if (a->batch <= 0 || a->seq <= 0 || a->n_kv_heads <= 0 || (a->head_dim != 64 && a->head_dim != 128) || a->max_ctx < a->seq ||
        (int64_t)a->batch * a->seq > 0x7fffffffLL || a->table_rows <= 0)
        return mi_fail(MI_E_SHAPE, "fill_cache: batch %d x %d tokens, %d heads of %d (64 or 128), a cache of %d", a->batch, a->seq, a->n_kv_heads, a->head_dim, a->max_ctx);
    if (a->dtype != MI_BF16 && a->dtype != MI_F16) return mi_fail(MI_E_DTYPE, "fill_cache: bf16 or f16 tensors (dtype code %d)", a->dtype);
    if (!a->k || !a->v || !a->k_rot || !a->k_cache || !a->v_cache || !a->ctx_len || !a->rotary_cos || !a->rotary_sin || !a->position_ids)
        return mi_fail(MI_E_NULL, "fill_cache: null pointer");
    if (!mi_aligned16(a->k) || !mi_aligned16(a->v) || !mi_aligned16(a->k_rot) || !mi_aligned16(a->k_cache) || !mi_aligned16(a->v_cache) ||
        !mi_aligned16(a->rotary_cos) || !mi_aligned16(a->rotary_sin))
        return mi_fail(MI_E_ALIGN, "fill_cache: tensors must be 16-byte aligned");
    for (const int64_t s : {a->k_stride_token, a->k_stride_head, a->v_stride_token, a->v_stride_head, a->cache_stride_batch, a->cache_stride_token, a->cache_stride_head})
        if (s % 8 != 0) return mi_fail(MI_E_ALIGN, "fill_cache: strides must be multiples of 8 elements");
    FillParams p{};
    p.k = a->k; p.v = a->v; p.cos = a->rotary_cos; p.sin = a->rotary_sin; p.pos = a->position_ids;
    p.k_out = a->k_rot; p.k_cache = a->k_cache; p.v_cache = a->v_cache; p.ctx_len = a->ctx_len;
    p.seq = a->seq; p.batch = a->batch; p.n_heads = a->n_kv_heads; p.n_tokens = (int64_t)a->batch * a->seq; p.table_rows = a->table_rows;
    p.k_st = a->k_stride_token; p.k_sh = a->k_stride_head; p.v_st = a->v_stride_token; p.v_sh = a->v_stride_head;
    p.c_sb = a->cache_stride_batch; p.c_st = a->cache_stride_token; p.c_sh = a->cache_stride_head;
    const int64_t items = p.n_tokens * a->n_kv_heads * (a->head_dim / 8), blocks = (items + kBlock - 1) / kBlock;     // more items than sequences
    if (items > 0xffffff00LL) return mi_fail(MI_E_SHAPE, "fill_cache: more than 2^32 vectors");
    const auto go = [&](auto t) {
        using T = decltype(t);
        const auto kernel = a->head_dim == 64 ? (a->rotary_interleaved ? fill_cache_kernel<T, 64, true> : fill_cache_kernel<T, 64, false>)
                                              : (a->rotary_interleaved ? fill_cache_kernel<T, 128, true> : fill_cache_kernel<T, 128, false>);
        kernel<<<dim3((unsigned)blocks), dim3(kBlock), 0, (hipStream_t)a->stream>>>(p);
    };
    if (a->dtype == MI_BF16) go(__bf16{});
    else go(_Float16{});
    return mi_check_launch("fill_cache");
}
