// sdpa_f32_fwd.hip -- fp32 Sdpa forward for gfx950, its products on the bf16
// matrix cores (sdpa_bf3.h).
//
// Replaces FlashAttnFwdKernel + FlashAttnFunctor<GPUDevice,float>
// (sdpa/sdpa_fwd.cu.cc:11-240); element semantics as in sdpa_fwd.hip.  A
// workgroup owns 128 queries of one batch row (four groups of 32, their
// parts in registers) and stages K/V blocks through registers into LDS, cut
// into their bf16 parts on the way, so that the four groups share the
// cutting; per 32 x 32 scores
//   S^T = K Q^T, online softmax, O^T += V^T P~^T  (P~ cut in registers).
// The keys of a tile may be divided over workgroups (fwd_f32_parts).
//
// What bounds it: VALU work (410 instructions per wave and 32 keys at
// 128/64: cutting, softmax) beside 72 MFMAs, which the two waves of a SIMD
// overlap only in part (the matrix cores are busy 52%).  B 64, S_q 512, D
// 128/64: 0.58 ms at 8192 keys, 0.89 ms on v_mfma_f32_32x32x2_f32 at 8224
// (73% busy; sdpa_f32_chain.hip, which takes over there), error against 64
// bits 1.1e-6 and 1.7e-6 (fewer roundings per sum); D 64: 0.41 and 0.65 ms.
// Not faster: staging one half of the waves earlier, operands read
// ahead, two workgroups of four waves per CU instead of one of eight.
#include <type_traits>

#include "sdpa_bf3.h"
#include "sdpa_launch.h"
#include "sdpa_merge.h"
#include "sdpa_params.h"
#include "sdpa_parts.h"

namespace sdpa {
namespace {

constexpr float kTau32 = 8.0f;  // lazy-rescale threshold (log2 units)

template <int DQK, int DV>
struct FwdBf3Cfg {
    // four query groups of 32 queries; NWK waves, on one SIMD, share each
    // group's keys (32 of a step's BN each) where registers and LDS allow
    static constexpr int NWK = DQK == 128 && DV == 128 ? 1 : 2, NT = 256 * NWK, BM = 128, BN = 32 * NWK;
    using KT = Bf3Tile<BN, DQK / 8>;
    using VT = Bf3Tile<BN, DV / 8>;
    static constexpr int STAGE = KT::BYTES + VT::BYTES;
    static constexpr int OS = DV + 4, MERGE = NWK > 1 ? (BM * OS + BM * 2) * 4 : 0;  // after the loop
    static constexpr size_t LDS_BYTES = 2 * STAGE > MERGE ? 2 * STAGE : MERGE;
    static_assert(LDS_BYTES <= 160 * 1024, "gfx950 LDS");
};

template <int DQK, int DV, bool VEC, bool DROP>
__global__ __launch_bounds__((FwdBf3Cfg<DQK, DV>::NT))
__attribute__((amdgpu_waves_per_eu(FwdBf3Cfg<DQK, DV>::NWK, FwdBf3Cfg<DQK, DV>::NWK)))
void sdpa_fwd_f32_bf3_kernel(const FwdParams p, const int win) {
    using Cfg = FwdBf3Cfg<DQK, DV>;
    using KT = typename Cfg::KT;
    using VT = typename Cfg::VT;
    constexpr int BM = Cfg::BM, BN = Cfg::BN, LK = DQK / 8, LV = DV / 8, NDT = DV / 32;

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

    const float* Qb = static_cast<const float*>(p.q) + (size_t)b * S_q * D_qk;
    const float* Kb = static_cast<const float*>(p.k) + (size_t)b * S_kv * D_qk;
    const float* Vb = static_cast<const float*>(p.v) + (size_t)b * S_kv * D_v;

    Bf3 q[DQK / 16];
    load_row_bf3<DQK, VEC>(q, Qb, my_q, S_q, D_qk, hh);
    prologue_loads_landed();
    // The running maximum is taken on raw scores, which needs a factor > 0:
    // for scale < 0 the queries are negated (their parts' signs), for scale 0
    // they are cleared.
    const float sl2 = p.c.scale_log2 == 0.f ? 1.f : fabsf(p.c.scale_log2);
    if (!(p.c.scale_log2 > 0.f)) {
        const uint32_t keep = p.c.scale_log2 == 0.f ? 0u : ~0u;
#pragma unroll
        for (int ks = 0; ks < DQK / 16; ++ks)
#pragma unroll
            for (int i = 0; i < 3; ++i) q[ks].p[i] = (q[ks].p[i] ^ 0x80008000u) & keep;
    }

    const int nblk = ((causal ? min(S_kv, q0 + BM) : S_kv) + BN - 1) / BN;
    const int lo = part_begin(nblk, part, np), hi = part_begin(nblk, part + 1, np);
    const bool wave_live = qw0 < S_q;
    const int wave_last_q = min(qw0 + 31, S_q - 1);
    floatx16 oacc[NDT];
    float m_run, l_run;
    const uint64_t st_base = DROP ? lcg_state(p.c.seed_offset, (uint64_t)b * S_q + my_q, (uint64_t)S_kv, 4 * hh) : 0;
    const uint32_t thr = p.c.drop_threshold;
    SwzLane<LK> swK;
    SwzLane<LV> swV;
    swK.init(lane);
    swV.init(lane);

    Bf3Stage<BN, DQK, Cfg::NT, VEC> kst;
    Bf3Stage<BN, DV, Cfg::NT, VEC> vst;
    auto load_block = [&](int blk) {
        const int n0 = blk * BN;
        kst.load(Kb, n0, S_kv - n0, D_qk, D_qk, tid);
        vst.load(Vb, n0, S_kv - n0, D_v, D_v, tid);
    };
    // INF: again, for infinities in V (sdpa_bf3.h).  Looking for them in V as it
    // is staged, or in the loop, cost 3 to 10%; the sums show them for nothing.
    auto pass = [&](auto inf) {
        constexpr bool INF = decltype(inf)::value;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) oacc[dt] = floatx16{};
        m_run = kMaxSentinel;
        l_run = 0.f;
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

        // The registers hold block blk + 1; it goes to LDS, and block blk + 2 into
        // the registers, at the end of the step.
        for (int blk = lo; blk < hi; ++blk) {
            const int kv0 = blk * BN + 32 * wk;
            const uint32_t ks0 = (uint32_t)(((blk - lo) & 1) * Cfg::STAGE), vs0 = ks0 + (uint32_t)KT::BYTES;
            if (wave_live && kv0 < S_kv && (!causal || kv0 <= wave_last_q)) {
                floatx16 s = floatx16{};
#pragma unroll
                for (int ks = 0; ks < DQK / 16; ++ks) s = mfma_bf3(KT::row(ks0 + swK.row, ks, 32 * wk), q[ks], s);
                if ((kv0 + 32 > S_kv) || (causal && kv0 + 31 > qw0)) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int key = kv0 + 8 * (r >> 2) + 4 * hh + (r & 3);
                        if (key >= S_kv || (causal && key > my_q)) s[r] = -INFINITY;
                    }
                }
                float mx = fmaxf(fmaxf(s[0], s[1]), s[2]);
#pragma unroll
                for (int r = 3; r < 15; r += 2) {
                    mx = fmaxf(mx, fmaxf(s[r], s[r + 1]));
                }
                mx = xhalf_max(fmaxf(mx, s[15])) * sl2;
                const float m_new = fmaxf(m_run, mx);
                if (wave_any(m_new > m_run + kTau32)) {
                    const float alpha = fast_exp2(m_run - m_new);
                    l_run *= alpha;
#pragma unroll
                    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                        for (int r = 0; r < 16; ++r) oacc[dt][r] *= alpha;
                    m_run = m_new;
                }
                const uint64_t st_blk = DROP ? st_base + (uint64_t)kv0 * kLcgMul : 0;
                float lsum = 0.f;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    s[r] = fast_exp2(__builtin_fmaf(s[r], sl2, -m_run));
                    lsum += s[r];
                }
                if (wave_any(lsum != lsum)) {
                    // A score of -inf (an infinite q or k) reads NaN in the sum of
                    // the parts' products, -inf in that of the first parts alone.
                    lds_read_again();
                    floatx16 h = floatx16{};
#pragma unroll
                    for (int ks = 0; ks < DQK / 16; ++ks)
                        h = mfma_bf16(KT::row(ks0 + swK.row, ks, 32 * wk).p[0], q[ks].p[0], h);
                    lsum = 0.f;
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        if (h[r] == -INFINITY) s[r] = 0.f;
                        lsum += s[r];
                    }
                }
                if constexpr (DROP) {
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        if (!lcg_keep(st_blk + (uint64_t)(8 * (r >> 2) + (r & 3)) * kLcgMul, thr)) s[r] = 0.f;
                }
                l_run += lsum;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const Bf3 pb = cut8([&](int i) { return s[8 * j + i]; });
                    Bf3 va[NDT];
#pragma unroll
                    for (int dt = 0; dt < NDT; ++dt) va[dt] = VT::tr(vs0 + swV.tr0, vs0 + swV.tr1, dt, 32 * wk + 16 * j);
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (INF) {
#pragma unroll
                        for (int dt = 0; dt < NDT; ++dt) oacc[dt] = mfma_bf3<true>(va[dt], pb, oacc[dt]);
                    } else {
#pragma unroll
                        for (int i = 0; i < 6; ++i)
#pragma unroll
                            for (int dt = 0; dt < NDT; ++dt) {
                                constexpr int ia[6] = {2, 0, 1, 1, 0, 0}, ib[6] = {0, 2, 1, 0, 1, 0};
                                oacc[dt] = mfma_bf16(va[dt].p[ia[i]], pb.p[ib[i]], oacc[dt]);
                            }
                    }
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
    if (workgroup_any_nan<Cfg::NT / 64>(oacc, tid)) pass(std::true_type{});

    float l_tot = xhalf_sum(l_run);
    if constexpr (Cfg::NWK == 2) {
        // O, m and l of the second wave of each group through LDS
        float* mo = reinterpret_cast<float*>(smem);
        float* ml = mo + BM * Cfg::OS;
        const int row = 32 * wq + l32;
        if (wk == 1) {
            store_rows_f32<DV, true>(mo + row * Cfg::OS, oacc, 1.f, hh, DV);
            if (hh == 0) {
                ml[2 * row] = m_run;
                ml[2 * row + 1] = l_tot;
            }
        }
        __syncthreads();
        if (wk == 1) return;
        const float m1 = ml[2 * row], M = fmaxf(m_run, m1), a0 = fast_exp2(m_run - M), a1 = fast_exp2(m1 - M);
        l_tot = l_tot * a0 + ml[2 * row + 1] * a1;
        m_run = M;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const floatx4 x = *reinterpret_cast<const floatx4*>(mo + row * Cfg::OS + 32 * dt + 8 * g + 4 * hh);
#pragma unroll
                for (int e = 0; e < 4; ++e) oacc[dt][4 * g + e] = oacc[dt][4 * g + e] * a0 + x[e] * a1;
            }
    }
    if (my_q < S_q && np > 1) {  // this part's unnormalised O, m and l
        const size_t at = (size_t)part * B * S_q + (size_t)b * S_q + my_q;
        if (hh == 0) {
            p.part_ml[2 * at] = m_run;
            p.part_ml[2 * at + 1] = l_tot;
        }
        store_rows_f32<DV, VEC>(p.part_o + at * D_v, oacc, 1.f, hh, D_v);
    } else if (my_q < S_q) {
        const float m_nat = (l_tot > 0.f) ? m_run * kLn2 : kNegInf;
        if (hh == 0) p.stats[(size_t)b * S_q + my_q] = m_nat + logf(l_tot + kEps);
        const float inv = (l_tot > kEps) ? p.c.keep_scale / l_tot : 0.f;
        store_rows_f32<DV, VEC>(static_cast<float*>(p.o) + ((size_t)b * S_q + my_q) * D_v, oacc, inv, hh, D_v);
    }
}

}  // namespace

hipError_t launch_fwd_f32(const FwdParams& p, bool vec, hipStream_t stream) {
    const int B = p.s.B, S_q = p.s.S_q;
    if (B == 0 || S_q == 0) return hipSuccess;
    if (fp32_chain_fwd(p.s, p.c.causal != 0)) return launch_fwd_f32_chain(p, vec, stream);
    return with_dim(p.s.D_qk, [&](auto dqk) {
        return with_dim(p.s.D_v, [&](auto dv) {
            return with_bool(vec, [&](auto v) {
                return with_bool(p.c.use_dropout != 0, [&](auto d) {
                    constexpr int DQK = decltype(dqk)::value, DV = decltype(dv)::value;
                    using Cfg = FwdBf3Cfg<DQK, DV>;
                    const long long n = (long long)((S_q + Cfg::BM - 1) / Cfg::BM) * p.parts * B;
                    const hipError_t err = launch_kernel<sdpa_fwd_f32_bf3_kernel<DQK, DV, decltype(v)::value, decltype(d)::value>>(
                        tile_grid(n, Cfg::NT), Cfg::NT, Cfg::LDS_BYTES, stream, p, row_window((size_t)p.s.S_kv * (DQK + DV) * 4));
                    return err == hipSuccess && p.parts > 1 ? launch_fwd_merge<float>(p, stream) : err;
                });
            });
        });
    });
}

}  // namespace sdpa
