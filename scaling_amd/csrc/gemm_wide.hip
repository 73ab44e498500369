// Matrix products of 16-bit types with 256 x 256 and 128 x 128 blocks: the projections of a layer, the LM head and their gradients.
// Same problems as gemm.hip (operands "rows" or "kmajor", up to three segments in one sum, several problems per launch).
//
// What bounds them is the matrix pipe and, with all compute units busy, the power it draws: a 8192^3 product that runs 2.0 PFLOP/s on zeros
// runs 1.5 on random numbers, and every byte an operand is moved costs time.  So
//   * a wavefront owns 128 x 128 (64 x 64) of the block, four such wavefronts per workgroup, one per SIMD: an operand fragment that is read from
//     LDS feeds eight (four) products.  Eight wavefronts of 128 x 64 read 1.5 x as much and run 0.78 ms where this runs 0.70;
//   * the products are v_mfma_*_16x16x32, whose accumulator traffic per multiply-add is half that of 32x32x16 (0.74 against 0.77 ms, the
//     same kernel with eight wavefronts);
//   * accumulators stay in accumulation registers for the whole kernel.  The products are inline assembly with such operands: left to
//     itself the compiler moves 64 tuples of four registers around in the loop (1.1 ms);
//   * tiles pass global -> LDS directly (buffer loads, so that whatever lies outside the matrix arrives as zero and steps past the
//     contraction cost no memory traffic), one and a half (three) steps of 64 ahead.  A half of a 256 x 256 x 64 stage is refilled as
//     soon as its fragments are in registers;
//   * reads and loads are spread evenly between the products (sched_barrier pins the order): with one wavefront per SIMD a clump of more
//     than three instructions between two products is a hole in the matrix pipe;
//   * with 16 steps of contraction a quarter of a block is what comes before and after them, so arguments come in two trips (ten, one after the other,
//     before), accumulators are cleared and the bias is fetched under the first tiles, and results are read, staged and stored a quadrant
//     at a time (all at once they did not fit the registers).  bf16, k 1024, before / after: 4084 x 4096 33.1 / 31.7 us, with bias 36.4 / 33.2;
//     4084 x 3072 with bias 34.0 / 30.7; 4084 x 1024 with bias, blocks of 128, 15.5 / 14.9; 8192 x 14336, k 4096 601 / 601.
// kmajor operands are read by LDS transpose reads from tiles in memory order, so all three layouts run at the same rate: 8192^3 bf16
// 0.70 / 0.71 / 0.71 ms (x W^T, dy W, dy^T x), the library 0.67 / 0.78 / 0.90 on the same box (another box: 0.71 / 0.72 / 0.73, 0.69 / 0.79 / 0.92).
//
// v_mfma_f32_16x16x32 operands, lane = 16 g + l:  A: row l, k = 8 g .. + 7;  B: column l, the same k;  C / D: column l, rows 4 g .. + 3.
// A = Q (output features), B = P (output rows): a lane holds four consecutive features of one output row.
#include "common.h"
#include "gemm_wide.h"

#include <algorithm>
#include <type_traits>

namespace {

typedef short v4i16_t __attribute__((ext_vector_type(4)));
typedef short v8i16_t __attribute__((ext_vector_type(8)));
typedef uint32_t srd_t __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int kStep = 64;                                  // contraction indices of a stage
constexpr int kBlockBytes = 64 * 128;                      // 64 x 64 elements
constexpr int kHalfBytes = 2 * kBlockBytes;                // 128 rows (columns) of one operand
constexpr int kStages128 = 4;
constexpr int kQBase = 65536;                              // P stages below, Q stages above

struct Segment { const char* p; const char* q; int64_t ldp, ldq; int k; };
struct Problem {
    int m, n, n_seg, p_kmajor, q_kmajor, first_block, tiles_m, tiles_n, splits, steps;
    uint32_t tiles_by, group_by;                           // for divide(): by tiles_m * tiles_n and kGroup * tiles_n
    Segment seg[MI_GEMM_MAX_SEGMENTS];
    void* c; const void* bias; const void* add;
    int64_t ldc, ldadd;
    float* part;                                           // splits > 1: fp32 partial results [splits][tiles_m * tile][tiles_n * tile]
    void* p_sum;                                           // column sums of a contraction-major P
    int sum_blocks;
};
struct Problems { int first_sum, first_block[MI_GEMM_MAX_PROBLEMS]; Problem p[MI_GEMM_MAX_PROBLEMS]; };   // no problem: first_block INT_MAX
// What a block needs before its first loads, and what it needs for its results
struct Block { Segment s; const void* bias; int m, n, n_seg, steps, splits; };
struct Out { void* c; const void* add; int64_t ldc, ldadd; int m, n; };
constexpr int kGroup = 4;                                  // block rows that are gone through together

#define PIN() __builtin_amdgcn_sched_barrier(0)

template <int N, int I = 0, class F> __device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<N, I + 1>(f);
    }
}

template <typename T> struct Half16;
template <> struct Half16<__bf16> {
    typedef bf16x8_t frag_t;
    static __device__ __forceinline__ void mma(f32x4_t& c, frag_t a, frag_t b) { asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b)); }
};
template <> struct Half16<_Float16> {
    typedef f16x8_t frag_t;
    static __device__ __forceinline__ void mma(f32x4_t& c, frag_t a, frag_t b) { asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b)); }
};

// Zeros that are in accumulation registers from here on: a compiler that wrote them right in front of the first product would leave out the two
// wait states between such a write and a product that reads it, as the products are inline assembly.
__device__ __forceinline__ void clear(f32x4_t& c) {
    c = f32x4_t{0.f, 0.f, 0.f, 0.f};
    asm volatile("" : "+a"(c));
}

// Results that are in accumulation registers up to here: left to itself the compiler reads all of them behind the last product, into registers that
// it has to clear first.
__device__ __forceinline__ f32x4_t fetch(f32x4_t c) {
    asm volatile("" : "+a"(c));
    return c;
}

// A 64 x 64 block in LDS: 64 rows (of the matrix as it lies in memory) of eight 16-byte units.  A direct load writes 64 x 16 consecutive
// bytes, so rows cannot be padded; the unit index of row r is XORed with swizzle(r) instead, which spreads the 16 rows that one pass of a
// 128-bit read touches over all banks, and likewise the four rows x 32 bytes of two lane groups of a transpose read.
__device__ __forceinline__ int swizzle(int r) { return (((r >> 1) & 1) << 2) | ((r >> 2) & 3); }

// Direct loads of one operand.  A step of 64 contraction indices of `HALVES` x 128 rows is HALVES x 16 instructions, four per wavefront and
// half.  The lane offsets are fixed, the bases of the buffer descriptors (one per half) move with the steps; their extents cover the present
// step's rows and columns only (so they never exceed 2^31 bytes) and are 0 past the end.
template <bool KMAJOR, int HALVES> struct Loader {
    uint32_t off[4];
    srd_t srd[HALVES];
    int step_bytes, left;                                  // contraction indices from the present step on, in this segment

    static __device__ __forceinline__ void source(int j, int wave, int lane, int& block, int& row, int& unit) {
        const int n = 4 * wave + j;
        block = n >> 3;
        row = 8 * (n & 7) + (lane >> 3);
        unit = (lane & 7) ^ swizzle(row);
    }
    __device__ __forceinline__ void open(const char* ptr, int64_t ld, int row0, int rows, int k, int wave, int lane) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            int block, r, u;
            source(j, wave, lane, block, r, u);
            off[j] = KMAJOR ? (uint32_t)(r * (int)ld * 2 + (block * 64 + 8 * u) * 2) : (uint32_t)((block * 64 + r) * (int)ld * 2 + u * 16);
        }
#pragma unroll
        for (int h = 0; h < HALVES; ++h) {
            const int first = row0 + h * 128, n = rows - first;
            const uint64_t base = (uint64_t)(ptr + (KMAJOR ? (int64_t)first * 2 : (int64_t)first * ld * 2));
            // columns of a kmajor operand in whole vectors: rows of it start on 16-byte boundaries
            const int extent = n <= 0 ? 0 : KMAJOR ? ((kStep - 1) * (int)ld + (n + 7) / 8 * 8) * 2 : ((min(n, 128) - 1) * (int)ld + kStep) * 2;
            srd[h][0] = __builtin_amdgcn_readfirstlane((uint32_t)base);
            srd[h][1] = __builtin_amdgcn_readfirstlane((uint32_t)(base >> 32) & 0xffffu);
            srd[h][2] = __builtin_amdgcn_readfirstlane(extent);
            srd[h][3] = 0x00020000u;
        }
        step_bytes = __builtin_amdgcn_readfirstlane(KMAJOR ? kStep * (int)ld * 2 : kStep * 2);
        left = k;
        if (left < kStep) last(wave, lane);
    }
    // The step that the contraction ends in.  Contiguous contraction indices end with a whole vector: an extent of an odd number of elements would
    // end inside the word that holds the last one.
    __device__ __forceinline__ void last(int wave, int lane) {
        const int cut = KMAJOR ? (kStep - left) * (step_bytes / kStep) : (kStep - (left + 7) / 8 * 8) * 2;
#pragma unroll
        for (int h = 0; h < HALVES; ++h) srd[h][2] = (uint32_t)max((int)srd[h][2] - cut, 0);
        if (!KMAJOR) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                int block, r, u;
                source(j, wave, lane, block, r, u);
                if (8 * u >= left) off[j] = 0xfffffff0u;
            }
        }
    }
    // to the next step; true: this segment has none
    __device__ __forceinline__ bool advance(int wave, int lane) {
#pragma unroll
        for (int h = 0; h < HALVES; ++h) {
            const uint64_t base = ((uint64_t)srd[h][0] | (uint64_t)srd[h][1] << 32) + (uint32_t)step_bytes;
            srd[h][0] = (uint32_t)base;
            srd[h][1] = (uint32_t)(base >> 32);
        }
        left -= kStep;
        if (left < kStep) {
            if (left <= 0) {
#pragma unroll
                for (int h = 0; h < HALVES; ++h) srd[h][2] = 0;
                return true;
            }
            last(wave, lane);
        }
        return false;
    }
    // instruction j of half h to LDS address dst + C; the completion is tracked by the explicit waits of the caller
    template <int C> __device__ __forceinline__ void load(int h, int j, uint32_t dst) const {
        asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(off[j]), "s"(srd[h]), "s"(dst), "n"(C)
                     : "memory", "m0", "scc");
    }
};

// Fragments of 16 rows t of a 64 x 64 block for contraction indices 32 ks ..
template <typename T, bool KMAJOR> struct Reader {
    using F = typename Half16<T>::frag_t;
    int b[4];
    __device__ __forceinline__ void init(int base, int lane) {
        const int l = lane & 15, g = lane >> 4;
        if (!KMAJOR) {
            b[0] = base + l * 128 + ((g ^ swizzle(l)) << 4);
            b[1] = base + l * 128 + (((4 + g) ^ swizzle(l)) << 4);
        } else {
            // transpose read: lane l of a group of 16 points at contraction row l / 4, columns 4 (l % 4) ..; rows 8 g .. + 3 and 8 g + 4 .. + 7
            const int r0 = 8 * g + (l >> 2), r1 = r0 + 4, e = (l >> 1) & 1, hb = l & 1;
            b[0] = base + r0 * 128 + ((e ^ swizzle(r0)) << 4) + 8 * hb;
            b[1] = base + r1 * 128 + ((e ^ swizzle(r1)) << 4) + 8 * hb;
            b[2] = b[0] ^ 64;
            b[3] = b[1] ^ 64;
        }
    }
    __device__ __forceinline__ F get(const char* smem, int off, int t, int ks) const {
        if constexpr (!KMAJOR) {
            return *reinterpret_cast<const F*>(smem + b[ks] + off + t * 2048);
        } else {
            typedef __attribute__((address_space(3))) v4i16_t lds_v4;
            const int x = (t & 1) << 5, o = off + ks * 4096;
            const char *lo = smem + (b[2 * (t >> 1)] ^ x) + o, *hi = smem + (b[2 * (t >> 1) + 1] ^ x) + o;
            const v4i16_t a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)(__attribute__((address_space(3))) void*)(void*)lo);
            const v4i16_t c = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)(__attribute__((address_space(3))) void*)(void*)hi);
            return __builtin_bit_cast(F, (v8i16_t)__builtin_shufflevector(a, c, 0, 1, 2, 3, 4, 5, 6, 7));
        }
    }
};

// The bias of a lane's features in 64 columns from n0 on.  Where four of them are a word of eight bytes they are requested in front of the tiles (and so
// are there with them); elsewhere when they are needed.
template <typename T> struct Bias {
    const T* at;                                           // nullable
    int n, n0;
    bool whole;
    uint2 raw[4];
    __device__ __forceinline__ void request(const Block& b, int first, int lane) {
        at = (const T*)b.bias;
        n = b.n;
        n0 = first + 4 * (lane >> 4);
        whole = at != nullptr && (n & 3) == 0 && ((uintptr_t)at & 7) == 0;
        if (whole) {
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) raw[nt] = *reinterpret_cast<const uint2*>(at + min(n0 + 16 * nt, n - 4));
        }
    }
    __device__ __forceinline__ f32x4_t get(int nt) const {
        f32x4_t x = {0.f, 0.f, 0.f, 0.f};
        if (whole) {
            typedef T t4 __attribute__((ext_vector_type(4)));
            const t4 v = __builtin_bit_cast(t4, raw[nt]);
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = (float)v[i];
        } else if (at != nullptr) {
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = Elem<T>::load1(at + min(n0 + 16 * nt + i, n - 1));
        }
        return x;
    }
};

// Results of a wavefront's 64 x 64 quadrant, with the bias, rounded, into 8 KB of LDS as rows.
template <typename T> __device__ __forceinline__ void stage_quadrant(const Bias<T>& bias, const f32x4_t (&acc)[4][4], char* stage, int lane) {
    typedef T t4 __attribute__((ext_vector_type(4)));
    const int l = lane & 15, g = lane >> 4;
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
        const f32x4_t add = bias.get(nt);
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            const int row = 16 * mt + l;
            const f32x4_t x = fetch(acc[mt][nt]);
            t4 v;
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = (T)(x[i] + add[i]);
            *reinterpret_cast<t4*>(stage + row * 128 + (((2 * nt + (g >> 1)) ^ swizzle(row)) << 4) + 8 * (g & 1)) = v;
        }
    }
}

// The staged rows to memory, eight lanes per row of 128 bytes.
template <typename T> __device__ __forceinline__ void store_quadrant(const Out& pr, const char* stage, int m0, int n0, int lane) {
    const int r8 = lane >> 3, u = lane & 7, n = n0 + 8 * u;
    const char* src = stage + r8 * 128;
    T* c = (T*)pr.c + (int64_t)(m0 + r8) * pr.ldc + n;
    if (pr.add == nullptr && m0 + 64 <= pr.m && n0 + 64 <= pr.n) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            *reinterpret_cast<u32x4_t*>(c + 8 * i * pr.ldc) = *reinterpret_cast<const u32x4_t*>(src + i * 1024 + ((u ^ swizzle(8 * i + r8)) << 4));
        return;
    }
    const T* add = (const T*)pr.add + (int64_t)(m0 + r8) * pr.ldadd + n;
#pragma unroll 2
    for (int i = 0; i < 8; ++i, c += 8 * pr.ldc, add += 8 * pr.ldadd) {
        if (m0 + r8 + 8 * i >= pr.m || n >= pr.n) continue;
        u32x4_t v = *reinterpret_cast<const u32x4_t*>(src + i * 1024 + ((u ^ swizzle(8 * i + r8)) << 4));
        if (n + 8 <= pr.n) {
            if (pr.add != nullptr) {                       // the product is rounded before it is added, as a separate product and sum would
                float x[8], y[8];
                Elem<T>::unpack(make_uint4(v[0], v[1], v[2], v[3]), x);
                Elem<T>::unpack(*reinterpret_cast<const uint4*>(add), y);
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] += y[e];
                const uint4 s = Elem<T>::pack(x);
                v = u32x4_t{s.x, s.y, s.z, s.w};
            }
            *reinterpret_cast<u32x4_t*>(c) = v;
        } else {
            const T* x = reinterpret_cast<const T*>(src + i * 1024 + ((u ^ swizzle(8 * i + r8)) << 4));
#pragma unroll 1
            for (int e = 0; e < pr.n - n; ++e) Elem<T>::store1(c + e, pr.add != nullptr ? Elem<T>::load1(x + e) + Elem<T>::load1(add + e) : Elem<T>::load1(x + e));
        }
    }
}

// A quadrant of a split's partial result: 16 rows of 64 bytes per store.
__device__ __forceinline__ void store_part(const Problem& pr, const f32x4_t (&acc)[4][4], int split, int tile, int m0, int n0, int lane) {
    const int64_t ld = (int64_t)pr.tiles_n * tile;
    float* c = pr.part + ((int64_t)split * pr.tiles_m * tile + m0 + (lane & 15)) * ld + n0 + 4 * (lane >> 4);
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) *reinterpret_cast<f32x4_t*>(c + 16 * mt * ld + 16 * nt) = fetch(acc[mt][nt]);
}

// Both operands of a problem, stepped together; a split of a problem (of one segment) takes the contraction indices k0 .. k0 + k - 1.
template <bool PK, bool QK, int HALVES> struct Operands {
    Loader<PK, HALVES> p;
    Loader<QK, HALVES> q;
    int seg, k0, k;
    __device__ __forceinline__ void open(const Segment& s, const Block& b, int m0, int n0, int wave, int lane) {
        const int len = b.splits > 1 ? k : s.k;
        p.open(s.p + (PK ? (int64_t)k0 * s.ldp : (int64_t)k0) * 2, s.ldp, m0, b.m, len, wave, lane);
        q.open(s.q + (QK ? (int64_t)k0 * s.ldq : (int64_t)k0) * 2, s.ldq, n0, b.n, len, wave, lane);
    }
    // returns the number of steps
    __device__ __forceinline__ int start(const Block& b, int split, int m0, int n0, int wave, int lane) {
        int steps = b.steps;
        seg = 0;
        k0 = 0;
        if (b.splits > 1) {
            const unsigned first = (unsigned)steps * split / b.splits, end = (unsigned)steps * (split + 1) / b.splits;
            k0 = first * kStep;
            k = min((int)end * kStep, b.s.k) - k0;
            steps = end - first;
        }
        open(b.s, b, m0, n0, wave, lane);
        return steps;
    }
    __device__ __forceinline__ void advance(const Problem& pr, const Block& b, int m0, int n0, int wave, int lane) {
        const bool end = p.advance(wave, lane);
        q.advance(wave, lane);
        if (end && seg + 1 < b.n_seg) {
            ++seg;
            open(pr.seg[seg], b, m0, n0, wave, lane);
        }
    }
};

// Requested between the first loads and the first products, not at the end.
__device__ __forceinline__ Out results(const Problem& pr, const Block& b) {
    Out out{pr.c, pr.add, pr.ldc, pr.ldadd, b.m, b.n};
    arrived(out.c, out.add, out.ldc, out.ldadd);
    return out;
}

template <int VM> __device__ __forceinline__ void wait_and_sync() {
    PIN();
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(VM) : "memory");
    PIN();
}
// of a wavefront whose loads are for nobody else
__device__ __forceinline__ void wait_and_sync() {
    PIN();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    PIN();
}

// 256 x 256: two stages, each of two halves per operand (rows 0 - 127 and 128 - 255; a wavefront takes 64 rows of each).  A step is four
// quadrants of 32 products in the order (A0, B0), (A0, B1), (A1, B1), (A1, B0), so that each brings one new half; fragments of the next
// half are read between the products of the present one, and the loads of step s + 2 go out as soon as a half's readers are through.  Two
// barriers per step, each a quarter of a quadrant after its boundary, where the reads before it have long completed.
template <typename T, bool PK, bool QK> __device__ __forceinline__ void tile256(const Problem& pr, const Block& blk, int split, int tm, int tn, char* smem) {
    using H = Half16<T>;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave >> 1, wn = wave & 1;
    const int m0 = tm * 256, n0 = tn * 256;
    const uint32_t dst = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem + wave * 4096);
    Operands<PK, QK, 2> in;
    const int steps = in.start(blk, split, m0, n0, wave, lane);
    Bias<T> bias[2];
    bias[0].request(blk, n0 + wn * 64, lane);
    bias[1].request(blk, n0 + 128 + wn * 64, lane);
    Reader<T, PK> rp;
    Reader<T, QK> rq;
    rp.init(wm * kBlockBytes, lane);
    rq.init(kQBase + wn * kBlockBytes, lane);
    f32x4_t acc[2][2][4][4];
    typename H::frag_t pf[2][4][2], qf[2][4][2];           // [half or set][16 rows][32 contraction indices]
    auto load_p = [&](auto s, auto h, auto j) { in.p.template load<s * 2 * kHalfBytes + h * kHalfBytes + j * 1024>(h, j, dst); PIN(); };
    auto load_q = [&](auto s, auto h, auto j) { in.q.template load<kQBase + s * 2 * kHalfBytes + h * kHalfBytes + j * 1024>(h, j, dst); PIN(); };
    auto read_p = [&](int s, int h, int f) { pf[h][f & 3][f >> 2] = rp.get(smem, (2 * s + h) * kHalfBytes, f & 3, f >> 2); PIN(); };
    auto read_q = [&](int set, int s, int h, int f) { qf[set][f & 3][f >> 2] = rq.get(smem, (2 * s + h) * kHalfBytes, f & 3, f >> 2); PIN(); };
    auto mma = [&](int h, int q, int set, int i) {         // one operand is the same for four products, the other for the turn of two rows
        const int ks = i >> 4, mt = (i >> 2) & 3, nt = (mt & 1) ? 3 - (i & 3) : (i & 3);
        H::mma(acc[h][q][mt][nt], qf[set][nt][ks], pf[h][mt][ks]);
        PIN();
    };
    static_for<2>([&](auto s) {
        static_for<2>([&](auto h) {
            static_for<4>([&](auto j) { load_q(s, h, j); });
            static_for<4>([&](auto j) { load_p(s, h, j); });
        });
        in.advance(pr, blk, m0, n0, wave, lane);
    });
    Out out = results(pr, blk);
    // while the first tiles are on their way
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int d = 0; d < 4; ++d) clear(acc[a][b][c][d]);
    wait_and_sync<24>();                                   // A0 and B0 of step 0
#pragma unroll
    for (int f = 0; f < 8; ++f) { read_q(0, 0, 0, f); read_p(0, 0, f); }
    auto step = [&](auto s_c) {
        constexpr int s = decltype(s_c)::value, X = s, Y = 1 - s;   // X holds B0, Y takes B1 and then the next B0
        constexpr std::integral_constant<int, 0> h0{};
        constexpr std::integral_constant<int, 1> h1{};
        static_for<32>([&](auto i) {
            if constexpr (i == 8) wait_and_sync<16>();     // A1, B1 of this step are there; A0, B0 are in everybody's registers
            mma(0, 0, X, i);
            if constexpr (i >= 8 && i % 3 == 2) read_q(Y, s, 1, i / 3 - 2);
            if constexpr (i >= 8 && i % 6 == 4) load_q(s_c, h0, std::integral_constant<int, i / 6 - 1>{});
        });
        static_for<32>([&](auto i) {
            mma(0, 1, Y, i);
            if constexpr (i % 4 == 1) read_p(s, 1, i / 4);
            if constexpr (i % 8 == 3) load_p(s_c, h0, std::integral_constant<int, i / 8>{});
        });
        static_for<32>([&](auto i) {
            if constexpr (i == 8) wait_and_sync<16>();     // A0, B0 of the next step are there; A1, B1 are in everybody's registers
            mma(1, 1, Y, i);
            if constexpr (i >= 8 && i % 3 == 2) read_p(1 - s, 0, i / 3 - 2);
            if constexpr (i >= 8 && i % 6 == 4) load_q(s_c, h1, std::integral_constant<int, i / 6 - 1>{});
        });
        static_for<32>([&](auto i) {
            mma(1, 0, X, i);
            if constexpr (i % 4 == 1) read_q(Y, 1 - s, 0, i / 4);
            if constexpr (i % 8 == 3) load_p(s_c, h1, std::integral_constant<int, i / 8>{});
            if constexpr (i == 30) in.advance(pr, blk, m0, n0, wave, lane);
        });
    };
    for (int i = 0; i < steps; i += 2) {                   // an odd count ends with a step of zeros
        step(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{});
    }
    asm volatile("s_nop 15" ::: "memory");                 // the last products' registers
    wait_and_sync<0>();
    if (blk.splits > 1) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int q = 0; q < 2; ++q) store_part(pr, acc[h][q], split, 256, m0 + h * 128 + wm * 64, n0 + q * 128 + wn * 64, lane);
        return;
    }
    // a quadrant is staged while the one before it is read back and stored
    const auto stage = [&](int i) { stage_quadrant<T>(bias[i & 1], acc[i >> 1][i & 1], smem + (4 * wave + i) * kBlockBytes, lane); };
    const auto store = [&](int i) {
        store_quadrant<T>(out, smem + (4 * wave + i) * kBlockBytes, m0 + (i >> 1) * 128 + wm * 64, n0 + (i & 1) * 128 + wn * 64, lane);
    };
    stage(0);
    PIN();
#pragma unroll
    for (int i = 1; i < 4; ++i) {
        stage(i);
        store(i - 1);
        PIN();
    }
    store(3);
}

// 128 x 128: four stages, loads three steps ahead, one barrier per step a quarter of its products after its start.  The fragments of the
// next step are read between the products of the present one.  Each of the four wavefronts has a neighbour on its SIMD that does nothing but load: a wavefront
// takes about 100 cycles to get rid of a direct load, and eight of them between 32 products of 16 cycles held the products up.  bf16, one wavefront
// per SIMD / two: 4084 x 1024, k 1024 with bias 15.2 / 13.8 us, k 4096 36.2 / 33.7; 2048 x 2048, k 8192 67.9 / 61.3; forward and backward of 4084 x 1024 -> 1024
// with bias 49.4 / 42.3.  (A fifth stage in place of the neighbour: level, 36.9 / 36.2.  A block of 256 has no registers for one.)
template <typename T, bool PK, bool QK> __device__ __forceinline__ void tile128(const Problem& pr, const Block& blk, int split, int tm, int tn, char* smem) {
    using H = Half16<T>;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 3, wm = wave >> 1, wn = wave & 1;
    const int m0 = tm * 128, n0 = tn * 128;
    Operands<PK, QK, 1> in;
    const int steps = in.start(blk, split, m0, n0, wave, lane);
    if (__builtin_amdgcn_readfirstlane(threadIdx.x) >= kThreads) {
        const uint32_t dst = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem + wave * 4096);
        const auto load = [&](int stage) {
            static_for<4>([&](auto j) { in.q.template load<kQBase + j * 1024>(0, j, dst + stage); });
            static_for<4>([&](auto j) { in.p.template load<j * 1024>(0, j, dst + stage); });
            in.advance(pr, blk, m0, n0, wave, lane);
        };
#pragma unroll
        for (int s = 0; s < kStages128; ++s) load(s * kHalfBytes);
        wait_and_sync<24>();                               // step 0
        for (int i = 0; i < (steps + 1) / 2 * 2; ++i) {
            wait_and_sync<16>();                           // the next step is there; the present one is in everybody's registers
            load((i & (kStages128 - 1)) * kHalfBytes);
        }
        wait_and_sync<0>();
        return;
    }
    Bias<T> bias;
    bias.request(blk, n0 + wn * 64, lane);
    Reader<T, PK> rp;
    Reader<T, QK> rq;
    rp.init(wm * kBlockBytes, lane);
    rq.init(kQBase + wn * kBlockBytes, lane);
    f32x4_t acc[4][4];
    typename H::frag_t pf[2][4][2], qf[2][4][2];           // [set][16 rows][32 contraction indices]
    auto read = [&](int set, int f, int stage) {           // the fragments of contraction indices 0 .. 31 first
        const int t = (f >> 1) & 3, ks = f >> 3;
        if (f & 1) pf[set][t][ks] = rp.get(smem + stage, 0, t, ks);
        else qf[set][t][ks] = rq.get(smem + stage, 0, t, ks);
        PIN();
    };
    auto mma = [&](int set, int i) {
        const int ks = i >> 4, mt = (i >> 2) & 3, nt = (mt & 1) ? 3 - (i & 3) : (i & 3);
        H::mma(acc[mt][nt], qf[set][nt][ks], pf[set][mt][ks]);
        PIN();
    };
    Out out = results(pr, blk);
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int d = 0; d < 4; ++d) clear(acc[c][d]);
    wait_and_sync();                                       // step 0
#pragma unroll
    for (int f = 0; f < 16; ++f) read(0, f, 0);
    int stage = 0;                                         // of the present step
    auto step = [&](auto x_c) {
        constexpr int X = decltype(x_c)::value, Y = 1 - X;
        const int next = (stage + kHalfBytes) & (kStages128 * kHalfBytes - 1);
        static_for<32>([&](auto i) {
            if constexpr (i == 8) wait_and_sync();
            mma(X, i);
            if constexpr (i >= 8 && i < 24) read(Y, i - 8, next);
        });
        stage = next;
    };
    for (int i = 0; i < steps; i += 2) {                   // an odd count ends with a step of zeros
        step(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{});
    }
    asm volatile("s_nop 15" ::: "memory");
    wait_and_sync();
    if (blk.splits > 1) {
        store_part(pr, acc, split, 128, m0 + wm * 64, n0 + wn * 64, lane);
        return;
    }
    stage_quadrant<T>(bias, acc, smem + wave * kBlockBytes, lane);
    store_quadrant<T>(out, smem + wave * kBlockBytes, m0 + wm * 64, n0 + wn * 64, lane);
}

// Bias gradients: sums over the rows of P, 64 columns per workgroup, behind the blocks of the products, where they run on compute units that
// the last round leaves idle and find most of P in the caches.  A launch of its own for each took 11 - 13 us at 4084 rows of 1024 .. 4096,
// with 16 .. 64 workgroups; here that is the cost only where the blocks are whole rounds (4084 x 4096 -> 1024, 75.7 -> 86.7 us), and nothing
// elsewhere (1024 -> 4096 86.6 -> 84.5, 1024 -> 3072 64.5 -> 64.6, 1024 -> 1024 35.2 -> 34.8).
constexpr int kSumColumns = 64;
template <typename T> __device__ __forceinline__ void sum_columns(const Problem& pr, int block, char* smem) {
    constexpr int V = 8, GROUPS = kThreads / 8, DEPTH = 8;
    const int lane = threadIdx.x & 63, u = threadIdx.x & 7, rows = pr.seg[0].k, col = block * kSumColumns + u * V;
    const int64_t ld = pr.seg[0].ldp;
    const T* base = (const T*)pr.seg[0].p + (col < pr.m ? col : 0);   // m is a whole number of vectors
    float acc[V];
#pragma unroll
    for (int i = 0; i < V; ++i) acc[i] = 0.f;
    const auto add = [&](const uint4& v) {
        float f[V];
        Elem<T>::unpack(v, f);
#pragma unroll
        for (int i = 0; i < V; ++i) acc[i] += f[i];
    };
    int r = threadIdx.x >> 3;
    for (; r + (DEPTH - 1) * GROUPS < rows; r += DEPTH * GROUPS) {
        uint4 v[DEPTH];
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) v[d] = *reinterpret_cast<const uint4*>(base + (int64_t)(r + d * GROUPS) * ld);
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) add(v[d]);
    }
    for (; r < rows; r += GROUPS) add(*reinterpret_cast<const uint4*>(base + (int64_t)r * ld));
#pragma unroll
    for (int i = 0; i < V; ++i) {
        acc[i] += __shfl_xor(acc[i], 8, MI_WAVE);
        acc[i] += __shfl_xor(acc[i], 16, MI_WAVE);
        acc[i] += __shfl_xor(acc[i], 32, MI_WAVE);
    }
    float* part = reinterpret_cast<float*>(smem);          // [wavefront][column]
    if (lane < 8) {
#pragma unroll
        for (int i = 0; i < V; ++i) part[(threadIdx.x >> 6) * kSumColumns + u * V + i] = acc[i];
    }
    __syncthreads();
    const int c = threadIdx.x;
    if (c < kSumColumns && block * kSumColumns + c < pr.m)
        Elem<T>::store1((T*)pr.p_sum + block * kSumColumns + c, (part[c] + part[kSumColumns + c]) + (part[2 * kSumColumns + c] + part[3 * kSumColumns + c]));
}

// Blocks of a problem are handed to the XCDs (workgroups modulo 8) in contiguous runs, in groups of four block rows, so that the workgroups
// that share an L2 read the same rows and columns at the same time.
template <typename T, int TILE>
__global__ __launch_bounds__(TILE == 256 ? kThreads : 2 * kThreads, TILE == 256 ? 1 : 2) void wide_kernel(const Problems ps) {
    __shared__ __attribute__((aligned(1024))) char smem[2 * kQBase];
    // Arguments in two trips, first which problem, then all that comes before the first loads: read where each is used they are ten in a row.
    int first_sum = ps.first_sum, i = 0;
    int first[MI_GEMM_MAX_PROBLEMS];
#pragma unroll
    for (int j = 1; j < MI_GEMM_MAX_PROBLEMS; ++j) first[j] = ps.first_block[j];
    arrived(first_sum, first[1], first[2], first[3], first[4], first[5]);
    static_assert(MI_GEMM_MAX_PROBLEMS == 6);
    if ((int)blockIdx.x >= first_sum) {
        if (TILE != 256 && threadIdx.x >= kThreads) return;
        int b = blockIdx.x - first_sum;
        while (b >= ps.p[i].sum_blocks) b -= ps.p[i++].sum_blocks;
        return sum_columns<T>(ps.p[i], b, smem);
    }
#pragma unroll
    for (int j = 1; j < MI_GEMM_MAX_PROBLEMS; ++j) i += (int)blockIdx.x >= first[j];
    const Problem& pr = ps.p[i];
    Block blk{pr.seg[0], pr.bias, pr.m, pr.n, pr.n_seg, pr.steps, pr.splits};
    int p_kmajor = pr.p_kmajor, q_kmajor = pr.q_kmajor, first_block = pr.first_block, tiles_m = pr.tiles_m, tiles_n = pr.tiles_n;
    uint32_t tiles_by = pr.tiles_by, group_by = pr.group_by;
    arrived(blk.s.p, blk.s.q, blk.s.ldp, blk.s.ldq, blk.s.k, blk.bias, blk.m, blk.n, blk.n_seg, blk.steps, blk.splits, p_kmajor, q_kmajor, first_block, tiles_m,
            tiles_n, tiles_by, group_by);
    const int tiles = tiles_m * tiles_n, total = tiles * blk.splits;
    const int b = blockIdx.x - first_block, xcd = b & 7, idx = b >> 3, each = total >> 3, rest = total & 7;
    if (idx >= each + (xcd < rest)) return;                // first_block is a multiple of eight
    const int item = xcd * each + min(xcd, rest) + idx, split = divide(item, tiles, tiles_by), t = item - split * tiles;
    const int per_group = kGroup * tiles_n, group = divide(t, per_group, group_by), row = group * kGroup, height = min(kGroup, tiles_m - row);
    const int in_group = t - group * per_group;
    const int tn = height == 4 ? in_group >> 2 : height == 3 ? divide(in_group, 3, 0x55555556u) : height == 2 ? in_group >> 1 : in_group;
    const int tm = row + in_group - tn * height;
    if constexpr (TILE == 256) {
        if (p_kmajor) tile256<T, true, true>(pr, blk, split, tm, tn, smem);
        else if (q_kmajor) tile256<T, false, true>(pr, blk, split, tm, tn, smem);
        else tile256<T, false, false>(pr, blk, split, tm, tn, smem);
    } else {
        if (p_kmajor) tile128<T, true, true>(pr, blk, split, tm, tn, smem);
        else if (q_kmajor) tile128<T, false, true>(pr, blk, split, tm, tn, smem);
        else tile128<T, false, false>(pr, blk, split, tm, tn, smem);
    }
}

// Sum of the partial results of a split problem in a fixed order, bias and residual as above: four features per thread.
template <typename T>
__global__ __launch_bounds__(256) void split_sum_kernel(const Problem pr, int tile) {
    const int groups = (pr.n + 3) / 4;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int m = (int)(i / groups), n = 4 * (int)(i - (int64_t)m * groups);
    if (m >= pr.m) return;
    const int64_t ld = (int64_t)pr.tiles_n * tile, stride = (int64_t)pr.tiles_m * tile * ld;
    const float* p = pr.part + (int64_t)m * ld + n;
    f32x4_t x = *reinterpret_cast<const f32x4_t*>(p);
    for (int s = 1; s < pr.splits; ++s) x += *reinterpret_cast<const f32x4_t*>(p + s * stride);
    T* c = (T*)pr.c + (int64_t)m * pr.ldc + n;
    const T* add = pr.add != nullptr ? (const T*)pr.add + (int64_t)m * pr.ldadd + n : nullptr;
    typedef T t4 __attribute__((ext_vector_type(4)));
    t4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int col = min(n + e, pr.n - 1);
        v[e] = (T)(pr.bias != nullptr ? x[e] + Elem<T>::load1((const T*)pr.bias + col) : x[e]);
        if (add != nullptr) v[e] = (T)((float)v[e] + Elem<T>::load1(add + col - n));
    }
    if (n + 4 <= pr.n) {
        *reinterpret_cast<t4*>(c) = v;
    } else {
        for (int e = 0; e < pr.n - n; ++e) c[e] = v[e];
    }
}

int steps_of(const mi_gemm_problem& a) {
    int steps = 0;
    for (int s = 0; s < a.n_segments; ++s) steps += (a.segments[s].k + kStep - 1) / kStep;
    return steps;
}
int64_t tiles_of(const mi_gemm_problem& a, int tile) { return (int64_t)((a.m + tile - 1) / tile) * ((a.n + tile - 1) / tile); }
double block_us(int tile, int steps) { return tile == 256 ? 7.5 + 1.3 * steps : 5.5 + 0.48 * steps; }

// A problem's first `at` rows (columns), or what follows them
mi_gemm_problem part(const mi_gemm_problem& a, bool columns, int at, bool first) {
    mi_gemm_problem r = a;
    if (first) {
        (columns ? r.n : r.m) = at;
        return r;
    }
    (columns ? r.n : r.m) -= at;
    for (int s = 0; s < a.n_segments; ++s) {
        auto& g = r.segments[s];
        if (columns) g.q = (const char*)g.q + 2 * (a.q_kmajor ? (int64_t)at : at * g.ldq);
        else g.p = (const char*)g.p + 2 * (a.p_kmajor ? (int64_t)at : at * g.ldp);
    }
    r.c = (char*)r.c + 2 * (columns ? (int64_t)at : at * r.ldc);
    if (r.add) r.add = (const char*)r.add + 2 * (columns ? (int64_t)at : at * r.ldadd);
    if (columns) {
        if (r.bias) r.bias = (const char*)r.bias + 2 * (int64_t)at;
        r.p_sum = nullptr;                                 // the first part has them all
    } else if (r.p_sum) {
        r.p_sum = (char*)r.p_sum + 2 * (int64_t)at;
    }
    return r;
}

// all problems but one; returns how many
int others(const mi_gemm_problem* in, int count, int but, mi_gemm_problem* out) {
    int n = 0;
    for (int i = 0; i < count; ++i)
        if (i != but) out[n++] = in[i];
    return n;
}

MiGemmPlan plan_in_one(const mi_gemm_problem* in, int count, size_t workspace_bytes, int cus);
int launch_in_one(const mi_gemm_problem* in, int count, int dtype, const MiGemmPlan& plan, void* workspace, hipStream_t st);

}  // namespace

// Blocks and splits by the time they are expected to take (us): a block costs `fixed` and `per_step` per step of 64, blocks come in rounds of
// one per compute unit, a split adds the traffic of its partial results and a launch.  Times that the figures come from, 128 / 256, bf16:
//   4084 x 1024, k 1024 13.4 / 25.2    4084 x 1024, k 4096 34.0 / 70.3    4084 x 4096, k 1024 47.7 / 32.5
//   2047 x 50257, k 1024 335 / 216     50257 x 1024, k 2047 283 / 198     2048 x 2048, k 2048 20.5 / 39.6    2048 x 5632, k 2048 56.3 / 43.3
namespace {
MiGemmPlan plan_in_one(const mi_gemm_problem* in, int count, size_t workspace_bytes, int cus) {
    MiGemmPlan best{};
    best.us = 1e30;
    for (int tile = 128; tile <= 256; tile += 128) {
        double work = 0, longest = 0, rounds_time = 0;
        int64_t tiles = 0;
        for (int i = 0; i < count; ++i) {
            const double t = block_us(tile, steps_of(in[i]));
            const int64_t n = tiles_of(in[i], tile);
            work += n * t;
            tiles += n;
            longest = t > longest ? t : longest;
        }
        // one problem: whole rounds; several: their blocks fill each other's gaps
        rounds_time = count == 1 ? longest * (double)((tiles + cus - 1) / cus) : (work / cus + (tiles > cus ? 0.5 * longest : 0));
        double us = rounds_time > longest ? rounds_time : longest;
        if (us < best.us) best = MiGemmPlan{us, tile, 1, 0, 0, false, 0};
        if (count == 1 && in[0].n_segments == 1) {
            const int steps = steps_of(in[0]);
            for (int s = 2; s <= 16 && tiles * s <= cus && steps / s >= 8; ++s) {
                const size_t bytes = (size_t)tiles * tile * tile * 4 * s;
                if (bytes > workspace_bytes) break;
                us = block_us(tile, (steps + s - 1) / s) + 3.0 + 2.0 * bytes / 5e6;
                if (us < best.us) best = MiGemmPlan{us, tile, s, bytes, 0, false, 0};
            }
        }
    }
    return best;
}

}  // namespace

// A problem whose last round is nearly empty goes in two launches: the rows or columns that make whole rounds, and the rest with a plan of its
// own.  It waits for the first to drain, so it has to promise 7 %.  Loss and gradients of an LM head, us: 2047 x 1024 x 50257 680 -> 652 (logits in
// 6 rounds and 160 small blocks instead of 7, weight gradient in 3 and 72 instead of 4), 8192 x 2048 x 9973 897 -> 820, 4096 x 4096 x 9973 level.
// Several problems go in one launch, where short blocks fill the gaps that long ones leave, unless one of them is a long chain of few blocks
// (tokens of a narrow layer: its weight gradient; few tokens before a wide output: its input gradient): it can be split over the chip only in a
// launch of its own.  All gradients, us, one launch / a launch each: 131072 x 256 -> 256 819 / 99, 32768 x 1024 -> 1024 213 / 131, 257 x 1024 ->
// 16384 97 / 43, 2090 x 1536 -> 128256 1906 / 1277, 1976 x 2048 -> 8192 142 / 113; 4084 x 1024 -> 4096 65 / 68, 300 x 4096 -> 14336 and 14336 273 / 352,
// 1468 x 4096 -> 4096 81 / 99.  A launch each is expected to take too little, mostly (of these 0.10, 0.45, 0.32, 0.57, 0.64 of one launch; 0.80, 0.80, 0.89), hence
// 0.65; the longest chain alone and the rest in one launch 0.70: 1024 x 4096 -> 14336 and 14336 573 / 476 (0.68), 32768 x 1024 -> three of 1024 425 / 430 (0.72).
MiGemmPlan mi_gemm_wide_plan(const mi_gemm_problem* in, int count, size_t workspace_bytes, int cus) {
    MiGemmPlan best = plan_in_one(in, count, workspace_bytes, cus);
    if (count > 1) {
        double each = 0, longest_us = 0;
        size_t bytes = 0, longest_bytes = 0;
        int longest = 0;
        for (int i = 0; i < count; ++i) {
            if (in[i].m == 0) continue;
            const MiGemmPlan p = mi_gemm_wide_plan(in + i, 1, workspace_bytes, cus);
            each += p.us;
            bytes = std::max(bytes, p.workspace_bytes);
            if (i > 0 && steps_of(in[i]) <= steps_of(in[longest])) continue;
            longest = i;
            longest_us = p.us;
            longest_bytes = p.workspace_bytes;
        }
        if (each < best.us * 0.65) return MiGemmPlan{each, 0, 1, bytes, 0, false, -1};
        mi_gemm_problem rest[MI_GEMM_MAX_PROBLEMS];
        const double two = longest_us + plan_in_one(rest, others(in, count, longest, rest), 0, cus).us;
        if (count > 2 && two < best.us * 0.70) return MiGemmPlan{two, 0, 1, longest_bytes, 0, false, longest + 1};
        return best;
    }
    const mi_gemm_problem& a = in[0];
    double us = best.us * 0.93;
    for (int tile = 128; tile <= 256; tile += 128) {
        const int64_t rounds = tiles_of(a, tile) / cus;
        if (rounds < 1) continue;
        for (int columns = 0; columns < 2; ++columns) {
            const int64_t across = ((columns ? a.m : a.n) + tile - 1) / tile, cut = rounds * cus / across * tile;
            if (cut < tile || cut >= (columns ? a.n : a.m)) continue;
            const mi_gemm_problem rest = part(a, columns, (int)cut, false);
            const MiGemmPlan p = plan_in_one(&rest, 1, workspace_bytes, cus);
            const double both = rounds * block_us(tile, steps_of(a)) + p.us;
            if (both < us) {
                us = both;
                best = MiGemmPlan{both, tile, 1, p.workspace_bytes, (int)cut, columns != 0, 0};
            }
        }
    }
    return best;
}

int mi_gemm_wide(const mi_gemm_problem* in, int count, int dtype, const MiGemmPlan& plan, void* workspace, int cus, hipStream_t st) {
    if (plan.apart != 0) {                                 // one after the other, with the same workspace
        int rc = MI_OK;
        for (int i = 0; i < count && rc == MI_OK; ++i)
            if (in[i].m > 0 && (plan.apart < 0 || plan.apart == i + 1))
                rc = mi_gemm_wide(in + i, 1, dtype, mi_gemm_wide_plan(in + i, 1, plan.workspace_bytes, cus), workspace, cus, st);
        if (plan.apart < 0 || rc != MI_OK) return rc;
        mi_gemm_problem rest[MI_GEMM_MAX_PROBLEMS];
        const int left = others(in, count, plan.apart - 1, rest);
        return launch_in_one(rest, left, dtype, plan_in_one(rest, left, 0, cus), nullptr, st);
    }
    if (plan.cut == 0) return launch_in_one(in, count, dtype, plan, workspace, st);
    const mi_gemm_problem first = part(in[0], plan.columns, plan.cut, true), rest = part(in[0], plan.columns, plan.cut, false);
    const int rc = launch_in_one(&first, 1, dtype, MiGemmPlan{plan.us, plan.tile, 1, 0, 0, false, 0}, nullptr, st);
    if (rc != MI_OK) return rc;
    return launch_in_one(&rest, 1, dtype, plan_in_one(&rest, 1, plan.workspace_bytes, cus), workspace, st);
}

namespace {
int launch_in_one(const mi_gemm_problem* in, int count, int dtype, const MiGemmPlan& plan, void* workspace, hipStream_t st) {
    const int tile = plan.tile;
    Problems ps;
    for (int& f : ps.first_block) f = 0x7fffffff;
    int order[MI_GEMM_MAX_PROBLEMS];
    for (int i = 0; i < count; ++i) {                      // longest contraction first: the launch then ends with short blocks
        int j = i;
        for (; j > 0 && steps_of(in[order[j - 1]]) < steps_of(in[i]); --j) order[j] = order[j - 1];
        order[j] = i;
    }
    int64_t total = 0;
    for (int i = 0; i < count; ++i) {
        const mi_gemm_problem& a = in[order[i]];
        Problem& p = ps.p[i];
        for (int s = 0; s < a.n_segments; ++s) {
            const auto& g = a.segments[s];
            p.seg[s] = Segment{(const char*)g.p, (const char*)g.q, g.ldp, g.ldq, g.k};
        }
        p.c = a.c; p.bias = a.bias; p.add = a.add; p.ldc = a.ldc; p.ldadd = a.ldadd; p.n_seg = a.n_segments;
        p.p_kmajor = a.p_kmajor; p.q_kmajor = a.q_kmajor; p.m = a.m; p.n = a.n;
        p.tiles_m = (a.m + tile - 1) / tile;
        p.tiles_n = (a.n + tile - 1) / tile;
        p.tiles_by = divide_m((uint32_t)(p.tiles_m * p.tiles_n));
        p.group_by = divide_m((uint32_t)(kGroup * p.tiles_n));
        p.steps = steps_of(a);
        p.splits = plan.splits;
        p.part = (float*)workspace;
        p.p_sum = a.p_sum;
        p.sum_blocks = a.p_sum != nullptr ? (a.m + kSumColumns - 1) / kSumColumns : 0;
        p.first_block = ps.first_block[i] = (int)total;
        total += ((int64_t)p.tiles_m * p.tiles_n * p.splits + 7) / 8 * 8;
        if (total > 0x7fffffffLL) return mi_fail(MI_E_SHAPE, "gemm: too many tiles");
    }
    ps.first_sum = (int)total;
    for (int i = 0; i < count; ++i) total += ps.p[i].sum_blocks;
    if (total == 0) return MI_OK;
    const dim3 grid((unsigned)total), block(kThreads);
    const Problem& p0 = ps.p[0];
    const dim3 sum_grid((unsigned)(((int64_t)p0.m * ((p0.n + 3) / 4) + 255) / 256));
    const auto go = [&](auto t) {
        using T = decltype(t);
        if (tile == 256) wide_kernel<T, 256><<<grid, block, 0, st>>>(ps);
        else wide_kernel<T, 128><<<grid, dim3(2 * kThreads), 0, st>>>(ps);
        if (plan.splits > 1) split_sum_kernel<T><<<sum_grid, block, 0, st>>>(p0, tile);
    };
    if (dtype == MI_BF16) go(__bf16{});
    else go(_Float16{});
    return mi_check_launch("gemm_wide");
}
}  // namespace
