// sdpa_f32_dq.hip -- fp32 SdpaGrad dQ kernel for gfx950 at D <= 64, its
// products on the bf16 matrix cores (sdpa_bf3.h), and the kernel that adds
// the parts of dQ, dK and dV where tiles are divided over workgroups.
//
// Replaces FlashAttnBwdKernel_Q for float (sdpa/sdpa_bwd.cu.cc:215-345);
// element semantics as in sdpa_bwd.hip.  128 queries per workgroup in four
// groups of 32; two waves, on one SIMD, share each group's keys (32 of a
// step's 64 each; their sums are added through LDS at the end).  K/V blocks
// are staged through registers into LDS, cut on the way.  A wider side needs
// more registers than two waves per SIMD have (Q, dO and dQ of 32 rows); the
// fp32 backward has its dS path there.  B 64, S_q 512, D 64: 0.51 ms at 8192
// keys, 0.99 ms on v_mfma_f32_32x32x2_f32 (sdpa_bwd.hip) at 8224, error against
// 64 bits 1.3e-6 and 1.8e-6.
#include <type_traits>

#include "sdpa_bf3.h"
#include "sdpa_launch.h"
#include "sdpa_params.h"
#include "sdpa_parts.h"

namespace sdpa {
namespace {

template <int DQK, int DV>
struct DqBf3Cfg {
    static constexpr int NT = 512, BM = 128, BN = 64;
    using KT = Bf3Tile<BN, DQK / 8>;
    using VT = Bf3Tile<BN, DV / 8>;
    static constexpr int STAGE = KT::BYTES + VT::BYTES;
    static constexpr int OS = DQK + 4, MERGE = BM * OS * 4;  // after the loop
    static constexpr size_t LDS_BYTES = 2 * STAGE > MERGE ? 2 * STAGE : MERGE;
    static_assert(LDS_BYTES <= 160 * 1024, "gfx950 LDS");
};

template <int DQK, int DV, bool VEC, bool DROP>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void sdpa_bwd_dq_f32_bf3_kernel(const BwdParams p, const int win) {
    using Cfg = DqBf3Cfg<DQK, DV>;
    using KT = typename Cfg::KT;
    using VT = typename Cfg::VT;
    constexpr int BM = Cfg::BM, BN = Cfg::BN, LK = DQK / 8, LV = DV / 8, NDT = DQK / 32;

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wq = wave & 3, wk = wave >> 2;
    const int B = p.s.B, S_q = p.s.S_q, S_kv = p.s.S_kv, D_qk = p.s.D_qk, D_v = p.s.D_v;
    const bool causal = p.c.causal != 0;
    const int np = p.parts, items = (S_q + BM - 1) / BM * np;
    int b, it;
    const int id = tile_id();
    if (id >= B * items) return;
    xcd_map(id, B * items, items, causal, win, b, it);
    const int qt = it / np, part = it - qt * np;
    const int q0 = qt * BM, qw0 = q0 + wq * 32, my_q = qw0 + l32;
    const size_t row_q = (size_t)b * S_q + my_q;

    const float* Ob = static_cast<const float*>(p.o) + (size_t)b * S_q * D_v;
    const float* dOb = static_cast<const float*>(p.d_o) + (size_t)b * S_q * D_v;
    const float* Kb = static_cast<const float*>(p.k) + (size_t)b * S_kv * D_qk;
    const float* Vb = static_cast<const float*>(p.v) + (size_t)b * S_kv * D_v;
    Bf3 q[DQK / 16], d_o[DV / 16];
    load_row_bf3<DQK, VEC>(q, static_cast<const float*>(p.q) + (size_t)b * S_q * D_qk, my_q, S_q, D_qk, hh);
    load_row_bf3<DV, VEC>(d_o, dOb, my_q, S_q, D_v, hh);
    float dpart = 0.f;
#pragma unroll
    for (int u = 0; u < DV / 8; ++u) {
        const int c = DV / 2 * hh + 4 * u;
        const floatx4 f = __builtin_bit_cast(floatx4, load_row_chunk<float, VEC>(dOb, my_q, S_q, c, D_v, D_v));
        const floatx4 o = __builtin_bit_cast(floatx4, load_row_chunk<float, VEC>(Ob, my_q, S_q, c, D_v, D_v));
#pragma unroll
        for (int e = 0; e < 4; ++e) dpart += f[e] * o[e];
    }
    const float delta = xhalf_sum(dpart);
    const bool row_ok = my_q < S_q;
    const float stats2 = row_ok ? p.stats[row_q] * kLog2e : INFINITY;
    if (row_ok && hh == 0 && wk == 0 && part == 0) {
        p.delta[row_q] = delta;
        p.stats2[row_q] = stats2 + kGateShift;
    }
    prologue_loads_landed();
    const float sl2 = p.c.scale_log2, ksc = p.c.keep_scale;

    const int nblk = ((causal ? min(S_kv, q0 + BM) : S_kv) + BN - 1) / BN;
    const int lo = part_begin(nblk, part, np), hi = part_begin(nblk, part + 1, np);
    const bool wave_live = qw0 < S_q;
    const int wave_last_q = min(qw0 + 31, S_q - 1);
    const uint64_t st_base = DROP ? lcg_state(p.c.seed_offset, row_q, (uint64_t)S_kv, 4 * hh) : 0;
    const uint32_t thr = p.c.drop_threshold;
    SwzLane<LK> swK;
    SwzLane<LV> swV;
    swK.init(lane);
    swV.init(lane);
    floatx16 dq[NDT];

    Bf3Stage<BN, DQK, Cfg::NT, VEC> kst;
    Bf3Stage<BN, DV, Cfg::NT, VEC> vst;
    auto load_block = [&](int blk) {
        const int n0 = blk * BN;
        kst.load(Kb, n0, S_kv - n0, D_qk, D_qk, tid);
        vst.load(Vb, n0, S_kv - n0, D_v, D_v, tid);
    };
    // INF: again, for infinities in V, dO or dS (sdpa_bf3.h)
    auto pass = [&](auto inf) {
        constexpr bool INF = decltype(inf)::value;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) dq[dt] = floatx16{};
        auto store_block = [&](int blk) {
            unsigned char* n = smem + ((blk - lo) & 1) * Cfg::STAGE;
            kst.store(n, tid);
            vst.template store<INF>(n + KT::BYTES, tid);
        };
        if (lo < hi) {
            load_block(lo);
            store_block(lo);
            if (lo + 1 < hi) load_block(lo + 1);
        }
        __syncthreads();

        for (int blk = lo; blk < hi; ++blk) {
            const int kv0 = blk * BN + 32 * wk;
            const uint32_t ks0 = (uint32_t)(((blk - lo) & 1) * Cfg::STAGE), vs0 = ks0 + (uint32_t)KT::BYTES;
            if (wave_live && kv0 < S_kv && (!causal || kv0 <= wave_last_q)) {
                floatx16 s = floatx16{}, dp = floatx16{};
#pragma unroll
                for (int ks = 0; ks < DQK / 16; ++ks) s = mfma_bf3(KT::row(ks0 + swK.row, ks, 32 * wk), q[ks], s);
#pragma unroll
                for (int ks = 0; ks < DV / 16; ++ks) dp = mfma_bf3<INF>(VT::row(vs0 + swV.row, ks, 32 * wk), d_o[ks], dp);
                float sum = 0.f;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    s[r] = fast_exp2(__builtin_fmaf(s[r], sl2, -stats2));
                    sum += s[r];
                }
                if (wave_any(sum != sum)) {  // scores of -inf (see sdpa_f32_fwd.hip)
                    lds_read_again();
                    floatx16 h = floatx16{};
#pragma unroll
                    for (int ks = 0; ks < DQK / 16; ++ks)
                        h = mfma_bf16(KT::row(ks0 + swK.row, ks, 32 * wk).p[0], q[ks].p[0], h);
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        if (h[r] * sl2 == -INFINITY) s[r] = 0.f;
                }
                if (kv0 + 32 > S_kv || (causal && kv0 + 31 > qw0)) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int key = kv0 + 8 * (r >> 2) + 4 * hh + (r & 3);
                        if (key >= S_kv || (causal && key > my_q)) s[r] = 0.f;
                    }
                }
                const uint64_t st_blk = DROP ? st_base + (uint64_t)kv0 * kLcgMul : 0;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float p0 = s[r] > kEps ? s[r] : 0.f;
                    float d = DROP ? dp[r] * ksc : dp[r];
                    if constexpr (DROP) d = lcg_keep(st_blk + (uint64_t)(8 * (r >> 2) + (r & 3)) * kLcgMul, thr) ? d : 0.f;
                    dp[r] = p0 * (d - delta);
                }
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const Bf3 ds = cut8<INF>([&](int i) { return dp[8 * j + i]; });
#pragma unroll
                    for (int dt = 0; dt < NDT; ++dt)
                        dq[dt] = mfma_bf3<INF>(KT::tr(ks0 + swK.tr0, ks0 + swK.tr1, dt, 32 * wk + 16 * j), ds, dq[dt]);
                }
            }
            if (blk + 1 < hi) {
                store_block(blk + 1);
                if (blk + 2 < hi) load_block(blk + 2);
            }
            __syncthreads();
        }
    };
    pass(std::false_type{});
    if (workgroup_any_nan<Cfg::NT / 64>(dq, tid)) pass(std::true_type{});

    // the second wave of each group through LDS
    float* m = reinterpret_cast<float*>(smem) + (32 * wq + l32) * Cfg::OS;
    if (wk == 1) store_rows_f32<DQK, true>(m, dq, 1.f, hh, DQK);
    __syncthreads();
    if (wk == 1 || !row_ok) return;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const floatx4 x = *reinterpret_cast<const floatx4*>(m + 32 * dt + 8 * g + 4 * hh);
#pragma unroll
            for (int e = 0; e < 4; ++e) dq[dt][4 * g + e] += x[e];
        }
    if (np > 1)
        store_rows_f32<DQK, VEC>(p.part_dq + ((size_t)part * B * S_q + row_q) * D_qk, dq, 1.f, hh, D_qk);
    else
        store_rows_f32<DQK, VEC>(static_cast<float*>(p.dq) + row_q * D_qk, dq, p.c.scale, hh, D_qk);
}

// dst[i] = f sum_k src[k n + i] over np parts, in part order; V values a thread.
struct SumJob {
    float* dst;
    const float* src;
    size_t n;
    int np;
    float f;
};
template <int V>
__device__ __forceinline__ void sum_parts(const SumJob& j, size_t i) {
    typedef float vec __attribute__((ext_vector_type(V)));
    vec s = vec{};
    constexpr int U = 4;  // loads in flight before the first is used
    for (int k0 = 0; k0 < j.np; k0 += U) {
        vec x[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
            x[u] = *reinterpret_cast<const vec*>(j.src + (size_t)(k0 + u < j.np ? k0 + u : j.np - 1) * j.n + i);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (k0 + u < j.np) s += x[u];
    }
    s *= j.f;
    if (((uintptr_t)(j.dst + i) & (sizeof(vec) - 1)) == 0) {
        *reinterpret_cast<vec*>(j.dst + i) = s;
    } else {
#pragma unroll
        for (int e = 0; e < V; ++e) j.dst[i + e] = s[e];
    }
}
template <int V>
__global__ __launch_bounds__(256) void sdpa_bwd_merge_f32_kernel(const SumJob a, const SumJob b, const SumJob c) {
    size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * V;
    if (i < a.n) return sum_parts<V>(a, i);
    i -= a.n;
    if (i < b.n) return sum_parts<V>(b, i);
    i -= b.n;
    if (i < c.n) sum_parts<V>(c, i);
}

}  // namespace

hipError_t launch_bwd_dq_f32(const BwdParams& p, bool vec, hipStream_t stream) {
    const int B = p.s.B, S_q = p.s.S_q;
    if (B == 0 || S_q == 0) return hipSuccess;
    return with_dim(p.s.D_qk, [&](auto dqk) {
        return with_dim(p.s.D_v, [&](auto dv) {
            return with_bool(vec, [&](auto v) {
                return with_bool(p.c.use_dropout != 0, [&](auto d) {
                    constexpr int DQK = decltype(dqk)::value, DV = decltype(dv)::value;
                    if constexpr (DQK <= 64 && DV <= 64) {
                        using Cfg = DqBf3Cfg<DQK, DV>;
                        const long long n = (long long)((S_q + Cfg::BM - 1) / Cfg::BM) * p.parts * B;
                        return launch_kernel<sdpa_bwd_dq_f32_bf3_kernel<DQK, DV, decltype(v)::value, decltype(d)::value>>(
                            tile_grid(n, Cfg::NT), Cfg::NT, Cfg::LDS_BYTES, stream, p, row_window((size_t)p.s.S_kv * (DQK + DV) * 4));
                    } else {
                        return hipErrorInvalidValue;
                    }
                });
            });
        });
    });
}

hipError_t launch_bwd_merge_f32(const BwdParams& p, hipStream_t stream) {
    const size_t rq = (size_t)p.s.B * p.s.S_q, rk = (size_t)p.s.B * p.s.S_kv;
    const SumJob none{nullptr, nullptr, 0, 0, 0.f};
    const SumJob q = p.parts > 1 ? SumJob{static_cast<float*>(p.dq), p.part_dq, rq * p.s.D_qk, p.parts, p.c.scale} : none;
    const SumJob k = p.kv_parts > 1 ? SumJob{static_cast<float*>(p.dk), p.part_dk, rk * p.s.D_qk, p.kv_parts, p.c.scale} : none;
    const SumJob v = p.kv_parts > 1 ? SumJob{static_cast<float*>(p.dv), p.part_dv, rk * p.s.D_v, p.kv_parts, p.c.keep_scale} : none;
    const size_t n = q.n + k.n + v.n;
    if (n == 0) return hipSuccess;
    if (p.s.D_qk % 4 == 0 && p.s.D_v % 4 == 0)
        return launch_kernel<sdpa_bwd_merge_f32_kernel<4>>((unsigned)((n / 4 + 255) / 256), 256, 0, stream, q, k, v);
    return launch_kernel<sdpa_bwd_merge_f32_kernel<1>>((unsigned)((n + 255) / 256), 256, 0, stream, q, k, v);
}

}  // namespace sdpa
