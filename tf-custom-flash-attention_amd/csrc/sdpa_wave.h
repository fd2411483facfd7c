// sdpa_wave.h -- pieces of the fp16 kernels for small grids, whose waves each
// stream tiles of their own through LDS (no barrier in the loop): a tile copy
// by one wave, the waits on it, and the sum of the waves' accumulators.
#pragma once

#include "sdpa_dma.h"

namespace sdpa {
namespace {

// Copies of one 32 x (8 L) fp16 tile by a single wave: copy u fills LDS chunk
// slots 64 u + lane, i.e. rows 64 u / L + lane / L.  The swizzle repeats every
// PERIOD copies (TR: the swz_tr layout of tiles read only transposed).
template <int L, bool TR>
struct WaveCopy {
    static constexpr int LOADS = L / 2, RPC = 64 / L;
    static constexpr int PERIOD = TR || RPC >= 16 ? 1 : 16 / RPC;
    static constexpr int NV = PERIOD < LOADS ? PERIOD : LOADS;
    uint32_t voff[NV];
    __device__ __forceinline__ void init(int lane, int row_bytes, int valid_chunks) {
#pragma unroll
        for (int u = 0; u < NV; ++u) {
            const int r = RPC * u + lane / L;
            const int c = (lane % L) ^ (TR ? swz_tr<L>(r) : swz<L>(r));
            voff[u] = c < valid_chunks ? (uint32_t)(r * row_bytes + c * 16) : kOob;
        }
    }
    __device__ __forceinline__ void issue(const RowSrc& src, uint32_t m0) const {
        const rsrc_t rs = src.at(0);
#pragma unroll
        for (int u = 0; u < LOADS; ++u)
            dma16_at(rs, m0 + 1024u * u, voff[u % NV] + (uint32_t)((u / NV) * NV * RPC * src.row_bytes));
    }
};

// s_waitcnt that the compiler does not move LDS reads across: the copies it
// waits for are invisible to it, and here no barrier follows.
template <int N>
__device__ __forceinline__ void wait_copies() {
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// Every LDS read of this wave has returned: its tile may be overwritten.
__device__ __forceinline__ void lds_reads_done() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// Row stride, in floats, of an accumulator of D features in LDS: 16 bytes
// off a whole number of bank rows, so that the lanes' rows spread over the banks.
constexpr int acc_stride(int D) { return D + 4; }

// The C^T accumulator of this lane's row (features 32 dt + 8 g + 4 hh + e)
// into row `row` of an LDS matrix of acc_stride(D) floats per row.
template <int D>
__device__ __forceinline__ void acc_to_lds(float* m, int row, const floatx16 (&acc)[D / 32], int hh) {
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *reinterpret_cast<floatx4*>(m + row * acc_stride(D) + 32 * dt + 8 * g + 4 * hh) =
                (floatx4){acc[dt][4 * g], acc[dt][4 * g + 1], acc[dt][4 * g + 2], acc[dt][4 * g + 3]};
}

// Sum over the NW waves of ROWS x D accumulators laid out by acc_to_lds (wave
// after wave, in that order); put(row, first column, four sums) for every
// four columns below ncols of the rows below nrows.
template <int NW, int ROWS, int D, typename Put>
__device__ __forceinline__ void sum_waves(const float* m, int tid, int nrows, int ncols, Put&& put) {
    constexpr int CPR = D / 4, N = ROWS * CPR, NT = 64 * NW;
#pragma unroll
    for (int i0 = 0; i0 < N; i0 += NT) {
        const int i = i0 + tid, row = i / CPR, c = 4 * (i % CPR);
        if ((N % NT != 0 && i >= N) || row >= nrows || c >= ncols) continue;
        floatx4 s = *reinterpret_cast<const floatx4*>(m + row * acc_stride(D) + c);
#pragma unroll
        for (int w = 1; w < NW; ++w) s += *reinterpret_cast<const floatx4*>(m + (w * ROWS + row) * acc_stride(D) + c);
        put(row, c, s);
    }
}

// Row operands of tiles whose feature size D is a multiple of 4 but not of 8
// (P4): the last chunk of a row, copied whole, ends in four features of the
// next row.  They only meet zeros of the other operand, but infinities there
// must not, so a reduction over features clears them; outputs past D are not
// stored.  keep4: which dwords 2 and 3 of chunk 2 ks + hh this lane keeps.
template <bool P4>
__device__ __forceinline__ half8 keep4(half8 x, int ks, int hh, int D) {
    if constexpr (P4) {
        typedef uint32_t u4 __attribute__((ext_vector_type(4)));
        u4 u = __builtin_bit_cast(u4, x);
        const uint32_t k = 16 * ks + 8 * hh + 4 < D ? ~0u : 0u;
        u[2] &= k;
        u[3] &= k;
        return __builtin_bit_cast(half8, u);
    }
    return x;
}

__device__ __forceinline__ half4 scaled_h4(const floatx4& s, float f) {
    half4 h;
#pragma unroll
    for (int e = 0; e < 4; ++e) h[e] = (half_t)(s[e] * f);
    return h;
}

}  // namespace
}  // namespace sdpa
