// sdpa_merge.h -- the forward's second kernel where a tile's keys are divided
// over workgroups (sdpa_parts.h).
#pragma once

#include "sdpa_device.h"
#include "sdpa_launch.h"
#include "sdpa_params.h"

namespace sdpa {
namespace {

// Merge of a row's parts: o = sum_i O_i 2^(m_i - M) / l, stats from M and l.
// One thread per four columns.
template <typename T>
__global__ __launch_bounds__(256) void sdpa_fwd_merge_kernel(const FwdParams p) {
    const int D_v = p.s.D_v, np = p.parts, cpr = (D_v + 3) / 4;
    const size_t rows = (size_t)p.s.B * p.s.S_q;
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const size_t row = i / cpr;
    const int c = 4 * (int)(i - row * cpr);
    if (row >= rows) return;
    // eight parts at a time: their loads all go out before the first is used
    // (one part after the other, each waited out the memory latency)
    constexpr int U = 8;
    float M = kMaxSentinel, L = 0.f;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < np; k0 += U) {
        float m[U], l[U], o[U][4];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u < np ? k0 + u : np - 1;
            const size_t at = k * rows + row;
            m[u] = p.part_ml[2 * at];
            l[u] = p.part_ml[2 * at + 1];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[u][e] = c + e < D_v ? p.part_o[at * D_v + c + e] : 0.f;
        }
        float Mn = M;
#pragma unroll
        for (int u = 0; u < U; ++u) Mn = fmaxf(Mn, m[u]);
        const float a = fast_exp2(M - Mn);
        L *= a;
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] *= a;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const float w = k0 + u < np ? fast_exp2(m[u] - Mn) : 0.f;
            L = __builtin_fmaf(l[u], w, L);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] = __builtin_fmaf(o[u][e], w, acc[e]);
        }
        M = Mn;
    }
    if (c == 0) p.stats[row] = ((L > 0.f) ? M * kLn2 : kNegInf) + logf(L + kEps);
    const float inv = (L > kEps) ? p.c.keep_scale / L : 0.f;
    T* o = static_cast<T*>(p.o) + row * D_v + c;
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (c + e < D_v) o[e] = (T)(acc[e] * inv);
}

template <typename T>
hipError_t launch_fwd_merge(const FwdParams& p, hipStream_t stream) {
    const long long th = (long long)p.s.B * p.s.S_q * ((p.s.D_v + 3) / 4);
    return launch_kernel<sdpa_fwd_merge_kernel<T>>((unsigned)((th + 255) / 256), 256, 0, stream, p);
}

}  // namespace
}  // namespace sdpa
