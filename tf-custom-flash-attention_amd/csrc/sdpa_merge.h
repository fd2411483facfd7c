// sdpa_merge.h -- the forward's second kernel where a tile's keys are divided
// over workgroups (sdpa_parts.h).
#pragma once

#include "sdpa_device.h"
#include "sdpa_launch.h"
#include "sdpa_params.h"

namespace sdpa {
namespace {

// Merge of a row's parts: o = sum_i O_i 2^(m_i - M) / l, stats from M and l.
// One thread per four columns; U parts at a time, whose loads all go out
// before the first is used (one part after the other, each waited out the
// memory latency).  V4: D_v is a multiple of 4.
template <typename T, int U, bool V4>
__global__ __launch_bounds__(256) void sdpa_fwd_merge_kernel(const FwdParams p) {
    const int D_v = p.s.D_v, np = p.parts, cpr = (D_v + 3) / 4;
    const size_t rows = (size_t)p.s.B * p.s.S_q;
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const size_t row = i / cpr;
    const int c = 4 * (int)(i - row * cpr);
    if (row >= rows) return;
    float M = kMaxSentinel, L = 0.f;
    floatx4 acc = floatx4{};
    for (int k0 = 0; k0 < np; k0 += U) {
        floatx2 ml[U];
        floatx4 o[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const size_t at = (k0 + u < np ? k0 + u : np - 1) * rows + row;
            ml[u] = *reinterpret_cast<const floatx2*>(p.part_ml + 2 * at);
            const float* src = p.part_o + at * D_v + c;
            if constexpr (V4) {
                o[u] = *reinterpret_cast<const floatx4*>(src);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) o[u][e] = c + e < D_v ? src[e] : 0.f;
            }
        }
        float Mn = M;
#pragma unroll
        for (int u = 0; u < U; ++u) Mn = fmaxf(Mn, ml[u][0]);
        const float a = fast_exp2(M - Mn);
        L *= a;
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] *= a;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k0 + u >= np) break;
            const float w = fast_exp2(ml[u][0] - Mn);
            L = __builtin_fmaf(ml[u][1], w, L);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] = __builtin_fmaf(o[u][e], w, acc[e]);
        }
        M = Mn;
    }
    if (c == 0) p.stats[row] = ((L > 0.f) ? M * kLn2 : kNegInf) + logf(L + kEps);
    const float inv = (L > kEps) ? p.c.keep_scale / L : 0.f;
    T* o = static_cast<T*>(p.o) + row * D_v + c;
    typedef T t4 __attribute__((ext_vector_type(4)));
    if constexpr (V4) {
        t4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (T)(acc[e] * inv);
        if (((uintptr_t)o & (sizeof(t4) - 1)) == 0) {
            *reinterpret_cast<t4*>(o) = v;
            return;
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (c + e < D_v) o[e] = (T)(acc[e] * inv);
}

template <typename T, int U>
hipError_t launch_fwd_merge_u(const FwdParams& p, unsigned n, hipStream_t stream) {
    if (p.s.D_v % 4 == 0) return launch_kernel<sdpa_fwd_merge_kernel<T, U, true>>(n, 256, 0, stream, p);
    return launch_kernel<sdpa_fwd_merge_kernel<T, U, false>>(n, 256, 0, stream, p);
}

template <typename T>
hipError_t launch_fwd_merge(const FwdParams& p, hipStream_t stream) {
    const unsigned n = (unsigned)(((long long)p.s.B * p.s.S_q * ((p.s.D_v + 3) / 4) + 255) / 256);
    if (p.parts <= 2) return launch_fwd_merge_u<T, 2>(p, n, stream);
    if (p.parts <= 4) return launch_fwd_merge_u<T, 4>(p, n, stream);
    return launch_fwd_merge_u<T, 8>(p, n, stream);
}

}  // namespace
}  // namespace sdpa
