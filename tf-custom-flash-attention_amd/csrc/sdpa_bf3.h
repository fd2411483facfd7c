// sdpa_bf3.h -- fp32 products on the bf16 matrix cores, for the fp32 kernels.
//
// v_mfma_f32_32x32x2_f32 runs at 1/16 of the bf16 rate on gfx950.  An fp32
// value is exactly the sum of three bf16 values (its top 8, next 8 and last
// 8 significant bits), so a product of two fp32 matrices is the sum of nine
// bf16 products with fp32 accumulation; the six of weight 2^-16 and above
//   lo hi, hi lo, mid mid, mid hi, hi mid, hi hi
// are taken (in that order, the small ones first), the three left out are
// below 2^-22 of |x||y| together.  Error against 64 bits, of the sum of the
// terms' magnitudes, largest and root mean square of 10^6 normal pairs, beside
// that of the fp32 chain: one term 2.4e-7 and 3.4e-8 (0.6e-7, 2.5e-8), four
// 1.9e-7 and 2.3e-8 (1.7e-7, 2.7e-8), sixteen 1.0e-7 and 1.3e-8 (2.3e-7,
// 2.8e-8): larger where one or two terms make the sum (a row that one weight
// dominates), smaller from four on.  Six products of 32x32x16 cost 6 x 32
// clocks where the fp32 form of the same reduction costs 8 x 64.
//
// The first part is cut off, not rounded: no part of a finite value
// overflows, and cutting takes an AND and an exact subtraction.  An infinite
// value leaves NaN parts, and without them would still be NaN times a small
// part of 0 or of the other sign.  A workgroup that finds a NaN in its sums
// at the end therefore goes over its tile again, with nothing below an infinity
// and infinities meeting first parts only (mfma_bf3<true>), which gives
// what the fp32 product gives.  Scores (Q and K) need less: one of -inf must
// weigh 0, which the kernels read from the product of the first parts; any
// other infinity in Q or K makes NaN in either form.
#pragma once

#include "sdpa_device.h"
#include "sdpa_dma.h"
#include "sdpa_tile.h"

namespace sdpa {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));
typedef uint32_t uint2v __attribute__((ext_vector_type(2)));

// Eight values of each part of an fp32 operand, hi first.
struct Bf3 {
    uint4v p[3];
};

__device__ __forceinline__ floatx16 mfma_bf16(const uint4v& a, const uint4v& b, const floatx16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
}
// w without its infinite halves
__device__ __forceinline__ uint32_t no_inf(uint32_t w) {
    const uint32_t l = (w & 0x7FFFu) == 0x7F80u ? 0xFFFF0000u : ~0u;
    const uint32_t h = (w & 0x7FFF0000u) == 0x7F800000u ? 0xFFFFu : ~0u;
    return w & l & h;
}
// c += A B over 16 reduction steps.  INF: operands may hold infinities (and
// are cut with INF).
template <bool INF = false>
__device__ __forceinline__ floatx16 mfma_bf3(const Bf3& a, const Bf3& b, floatx16 c) {
    if constexpr (INF) {
        uint4v a0, b0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            a0[i] = no_inf(a.p[0][i]);
            b0[i] = no_inf(b.p[0][i]);
        }
        c = mfma_bf16(a.p[2], b0, c);
        c = mfma_bf16(a0, b.p[2], c);
        c = mfma_bf16(a.p[1], b.p[1], c);
        c = mfma_bf16(a.p[1], b0, c);
        c = mfma_bf16(a0, b.p[1], c);
        return mfma_bf16(a.p[0], b.p[0], c);
    }
    c = mfma_bf16(a.p[2], b.p[0], c);
    c = mfma_bf16(a.p[0], b.p[2], c);
    c = mfma_bf16(a.p[1], b.p[1], c);
    c = mfma_bf16(a.p[1], b.p[0], c);
    c = mfma_bf16(a.p[0], b.p[1], c);
    return mfma_bf16(a.p[0], b.p[0], c);
}

// Whether an accumulator of the workgroup's NW waves holds a NaN, which an
// infinite factor leaves there for certain.  (Sums past 1e19 may answer yes as
// well, which costs time only.)  LDS is free before (a barrier ago) and after.
template <int NW, int N>
__device__ __forceinline__ bool workgroup_any_nan(const floatx16 (&acc)[N], int tid) {
    float z = 0.f;
#pragma unroll
    for (int dt = 0; dt < N; ++dt)
#pragma unroll
        for (int r = 0; r < 16; r += 2) z = __builtin_fmaf(acc[dt][r], acc[dt][r + 1], z);
    const bool mine = wave_any(!(__builtin_fabsf(z) < INFINITY));
    uint32_t* slot = reinterpret_cast<uint32_t*>(smem);
    if ((tid & 63) == 0) slot[tid >> 6] = mine;
    __syncthreads();
    uint32_t all = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) all |= slot[w];
    __syncthreads();
    return __builtin_amdgcn_readfirstlane((int)all) != 0;
}

// Upper halves of two dwords, a's below b's.
__device__ __forceinline__ uint32_t pack_hi16(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }

// Two values rounded to bf16 (to nearest even), a in the low half.
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){a, b}, b2));
}

// The parts of two values, packed (a in the low half): hi cut off, mid
// rounded (so that lo, which the dropped products carry, has no bias), lo
// what is left, exactly.  INF: an infinite value has mid = lo = 0.
template <bool INF = false>
__device__ __forceinline__ void cut2(float a, float b, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
    const uint32_t ua = __float_as_uint(a), ub = __float_as_uint(b);
    hi = pack_hi16(ua, ub);
    float ra = a - __uint_as_float(ua & 0xFFFF0000u), rb = b - __uint_as_float(ub & 0xFFFF0000u);
    if constexpr (INF) {
        if ((ua & 0x7FFFFFFFu) == 0x7F800000u) ra = 0.f;
        if ((ub & 0x7FFFFFFFu) == 0x7F800000u) rb = 0.f;
    }
    mid = pack_bf16(ra, rb);
    lo = pack_hi16(__float_as_uint(ra - __uint_as_float(mid << 16)),
                   __float_as_uint(rb - __uint_as_float(mid & 0xFFFF0000u)));
}
// Parts of eight values (two of them per dword, in order).
template <bool INF = false, typename Get>
__device__ __forceinline__ Bf3 cut8(Get&& x) {
    Bf3 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t h, m, l;
        cut2<INF>(x(2 * i), x(2 * i + 1), h, m, l);
        r.p[0][i] = h;
        r.p[1][i] = m;
        r.p[2][i] = l;
    }
    return r;
}

// What was read from LDS is read again after this: the rare repair of scores
// does not keep the loop's operands in registers.
__device__ __forceinline__ void lds_read_again() { asm volatile("" ::: "memory"); }

// A ROWS x (8 L) tile in LDS as three planes of PLANE bytes (hi, mid, lo),
// each in the chunk-swizzled layout of swz_off.
template <int ROWS, int L>
struct Bf3Tile {
    static constexpr int PLANE = ROWS * L * 16, BYTES = 3 * PLANE;
    // the parts of four consecutive values, columns col .. col + 3 (col % 4 == 0)
    template <bool INF>
    __device__ __forceinline__ static void store4(unsigned char* tile, int row, int col, const floatx4& v) {
        uint32_t h[2], m[2], l[2];
        cut2<INF>(v[0], v[1], h[0], m[0], l[0]);
        cut2<INF>(v[2], v[3], h[1], m[1], l[1]);
        unsigned char* d = tile + 2 * swz_off<L>(row, col);
        *reinterpret_cast<uint2v*>(d) = (uint2v){h[0], h[1]};
        *reinterpret_cast<uint2v*>(d + PLANE) = (uint2v){m[0], m[1]};
        *reinterpret_cast<uint2v*>(d + 2 * PLANE) = (uint2v){l[0], l[1]};
    }
    // A operand, rows R0 + l32, features 16 ks + 8 hh ..; a = tile offset + SwzLane::row
    __device__ __forceinline__ static Bf3 row(uint32_t a, int ks, int R0) {
        Bf3 r;
#pragma unroll
        for (int i = 0; i < 3; ++i) r.p[i] = __builtin_bit_cast(uint4v, lds_row<L>(a + i * PLANE, ks, R0));
        return r;
    }
    // Transposed A operand (lds_tr); a0 / a1 = tile offset + SwzLane::tr0 / tr1
    __device__ __forceinline__ static Bf3 tr(uint32_t a0, uint32_t a1, int dt, int R0) {
        Bf3 r;
#pragma unroll
        for (int i = 0; i < 3; ++i) r.p[i] = __builtin_bit_cast(uint4v, lds_tr<L>(a0 + i * PLANE, a1 + i * PLANE, dt, R0));
        return r;
    }
};

// A tile staged through registers (TileStage) into a Bf3Tile.
template <int ROWS, int COLS, int NTHREADS, bool VEC>
struct Bf3Stage {
    TileStage<float, ROWS, COLS, NTHREADS, VEC> t;
    __device__ __forceinline__ void load(const float* g, int row0, int nrows, int ncols, int ld, int tid) {
        t.load(g, row0, nrows, ncols, ld, tid);
    }
    template <bool INF = false>
    __device__ __forceinline__ void store(unsigned char* tile, int tid) const {
        using S = TileStage<float, ROWS, COLS, NTHREADS, VEC>;
#pragma unroll
        for (int u = 0; u < S::PER_THREAD; ++u) {
            const int c = tid + u * NTHREADS;
            if (S::NCH % NTHREADS == 0 || c < S::NCH)
                Bf3Tile<ROWS, COLS / 8>::template store4<INF>(tile, c / S::CPR, (c % S::CPR) * 4,
                                                             __builtin_bit_cast(floatx4, t.r[u]));
        }
    }
};

// B operand of one row (lane = row, features 16 ks + 8 hh .. + 7), with nothing
// below an infinity.
template <int D, bool VEC>
__device__ __forceinline__ void load_row_bf3(Bf3 (&r)[D / 16], const float* g, int row, int nrows, int ncols, int hh) {
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
        const int c = 16 * ks + 8 * hh;
        const floatx4 x = __builtin_bit_cast(floatx4, load_row_chunk<float, VEC>(g, row, nrows, c, ncols, ncols));
        const floatx4 y = __builtin_bit_cast(floatx4, load_row_chunk<float, VEC>(g, row, nrows, c + 4, ncols, ncols));
        r[ks] = cut8<true>([&](int i) { return i < 4 ? x[i] : y[i - 4]; });
    }
}

// Store the C^T accumulator of this lane's output row (features 32 dt + 8 g +
// 4 hh + e) times f; columns from ncols on are not written.
template <int D, bool VEC>
__device__ __forceinline__ void store_rows_f32(float* dst, const floatx16 (&acc)[D / 32], float f, int hh, int ncols) {
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int d0 = 32 * dt + 8 * g + 4 * hh;
            floatx4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = acc[dt][4 * g + e] * f;
            if constexpr (VEC) {
                if (d0 < ncols) *reinterpret_cast<floatx4*>(dst + d0) = v;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (d0 + e < ncols) dst[d0 + e] = v[e];
            }
        }
}

}  // namespace
}  // namespace sdpa
