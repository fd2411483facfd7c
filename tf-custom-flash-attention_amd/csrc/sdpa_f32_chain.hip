// sdpa_f32_chain.hip -- the fp32 forward and dK/dV on
// v_mfma_f32_32x32x2_f32, for the shapes of fp32_chain_fwd() and fp32_chain() (sdpa_parts.h); all
// others run on the bf16 matrix cores (sdpa_f32_fwd.hip, sdpa_f32_dkdv.hip).
//
// The gradient leaves out weights P <= 1e-6, a step, and a weight within a
// rounding of it (4e-6 of it, measured) goes one way or the other with the
// order in which its score and its row's stats were summed.  From about 16384
// keys on that step lies among the weights of ordinary rows.  Against these
// kernels the bf16-part ones moved a weight across it, which changes an element
// of dK or dV by 1e-3 to 9e-3 of their root mean square, in 6 of 10 calls at
// B 64, S_q 512, S_kv 16384, D 128/64, in 1 of 6 at D 64/64 and in 3 of 8 at
// B 16, S_q 100, D 80; in none of 8 at B 64, S_q 256, S_kv 12000, and in none
// of 32 at 2048 to 8192 keys.  Neither side is the more exact one; these
// shapes keep the side that they had.  It costs time: the first shape's
// forward takes 1.76 ms here, 1.08 there, its dK/dV 3.53, 2.50 there.
// What bounds both here: the fp32 matrix rate, 75% busy.
//
// Feature reductions are split between the half-waves: lane-half h covers
// features [h D/2, (h+1) D/2), so operands are read as float4 runs;
// reductions over keys or queries pair k-step r of lane-half h with row 8
// (r/4) + 4h + r%4 of the 32-row accumulator tile.
//
// The forward serves few keys against many tiles as well, where it is the faster
// one (fp32_chain_fwd()).
#include <type_traits>

#include "sdpa_dma.h"
#include "sdpa_launch.h"
#include "sdpa_params.h"

namespace sdpa {
namespace {

constexpr float kTauChain = 8.0f;  // lazy-rescale threshold (log2 units)

// Workgroup -> (batch, tile), level-major; reversed (heaviest first) for
// causal query tiles.
__device__ __forceinline__ void map_q_tile(int bid, int B, int tiles, bool causal, int& b, int& t) {
    b = bid % B;
    const int level = bid / B;
    t = causal ? (tiles - 1 - level) : level;
}


// ---------------------------------------------------------------------------
// Forward: 128 queries per workgroup, K/V blocks of 32 keys staged through
// registers into two LDS stages.
// ---------------------------------------------------------------------------
template <int DQK, int DV>
struct FwdChainCfg {
    static constexpr int NT = 256, BM = 128, BN = 32;
    static constexpr int KS = DQK + 4;  // float4 reads by 16 rows hit 64 distinct banks
    static constexpr int VS = DV + 8;   // the two half-waves read rows 4 apart: disjoint banks
    static constexpr int KT = BN * KS, VT = BN * VS, STAGE = KT + VT;
    static constexpr size_t LDS_BYTES = 2 * (size_t)STAGE * sizeof(float);
};

template <int DQK, int DV, bool VEC, bool DROP>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void sdpa_fwd_f32_chain_kernel(const FwdParams p) {
    using Cfg = FwdChainCfg<DQK, DV>;
    constexpr int BM = Cfg::BM, BN = Cfg::BN, KS = Cfg::KS, VS = Cfg::VS;
    constexpr int HQ = DQK / 2;  // features per half-wave
    float* lds = reinterpret_cast<float*>(smem);

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l32 = lane & 31, hh = lane >> 5;
    const int B = p.s.B, S_q = p.s.S_q, S_kv = p.s.S_kv, D_qk = p.s.D_qk, D_v = p.s.D_v;
    const bool causal = p.c.causal != 0;
    const int tiles = (S_q + BM - 1) / BM;
    int b, qt;
    map_q_tile(blockIdx.x, B, tiles, causal, b, qt);
    const int q0 = qt * BM, qw0 = q0 + wave * 32, my_q = qw0 + l32;

    const float* Qb = static_cast<const float*>(p.q) + (size_t)b * S_q * D_qk;
    const float* Kb = static_cast<const float*>(p.k) + (size_t)b * S_kv * D_qk;
    const float* Vb = static_cast<const float*>(p.v) + (size_t)b * S_kv * D_v;

    float qf[HQ];
#pragma unroll
    for (int u = 0; u < HQ / 4; ++u) {
        const uint4 c = load_row_chunk<float, VEC>(Qb, my_q, S_q, HQ * hh + 4 * u, D_qk, D_qk);
        const floatx4 f = __builtin_bit_cast(floatx4, c);
#pragma unroll
        for (int e = 0; e < 4; ++e) qf[4 * u + e] = f[e];
    }
    prologue_loads_landed();

    const int kv_end = causal ? min(S_kv, q0 + BM) : S_kv;
    const int nblk = (kv_end + BN - 1) / BN;
    const bool wave_live = qw0 < S_q;
    const int wave_last_q = min(qw0 + 31, S_q - 1);

    floatx16 oacc[DV / 32];
#pragma unroll
    for (int dt = 0; dt < DV / 32; ++dt) oacc[dt] = floatx16{};
    float m_run = kMaxSentinel, l_run = 0.f;
    const float sl2 = p.c.scale_log2;
    const uint64_t st_base =
        DROP ? lcg_state(p.c.seed_offset, (uint64_t)b * S_q + my_q, (uint64_t)S_kv, 4 * hh) : 0;
    const uint32_t thr = p.c.drop_threshold;

    TileStage<float, BN, DQK, Cfg::NT, VEC> kst;
    TileStage<float, BN, DV, Cfg::NT, VEC> vst;
    if (nblk > 0) {
        kst.load(Kb, 0, S_kv, D_qk, D_qk, tid);
        vst.load(Vb, 0, S_kv, D_v, D_v, tid);
        kst.template store<KS>(lds, tid);
        vst.template store<VS>(lds + Cfg::KT, tid);
    }
    __syncthreads();

    for (int blk = 0; blk < nblk; ++blk) {
        const int kv0 = blk * BN;
        const float* Ks = lds + (blk & 1) * Cfg::STAGE;
        const float* Vs = Ks + Cfg::KT;
        const bool has_next = blk + 1 < nblk;
        if (has_next) {
            kst.load(Kb, kv0 + BN, S_kv - kv0 - BN, D_qk, D_qk, tid);
            vst.load(Vb, kv0 + BN, S_kv - kv0 - BN, D_v, D_v, tid);
        }

        if (wave_live && (!causal || kv0 <= wave_last_q)) {
            floatx16 sacc = floatx16{};
#pragma unroll
            for (int u = 0; u < HQ / 4; ++u) {
                const floatx4 kk = *reinterpret_cast<const floatx4*>(Ks + l32 * KS + HQ * hh + 4 * u);
#pragma unroll
                for (int e = 0; e < 4; ++e) sacc = mfma_f32(kk[e], qf[4 * u + e], sacc);
            }
            const bool need_mask = (kv0 + BN > S_kv) || (causal && kv0 + BN - 1 > qw0);
            float mx = -INFINITY;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                float x = sacc[r] * sl2;
                if (need_mask) {
                    const int key = kv0 + 8 * (r >> 2) + 4 * hh + (r & 3);
                    if (key >= S_kv || (causal && key > my_q)) x = -INFINITY;
                }
                sacc[r] = x;
                mx = fmaxf(mx, x);
            }
            mx = xhalf_max(mx);
            const float m_new = fmaxf(m_run, mx);
            if (wave_any(m_new > m_run + kTauChain)) {
                const float alpha = fast_exp2(m_run - m_new);
                l_run *= alpha;
#pragma unroll
                for (int dt = 0; dt < DV / 32; ++dt)
#pragma unroll
                    for (int r = 0; r < 16; ++r) oacc[dt][r] *= alpha;
                m_run = m_new;
            }
            const uint64_t st_blk = DROP ? st_base + (uint64_t)kv0 * kLcgMul : 0;
            float lsum = 0.f;
            float pr[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                float pv = fast_exp2(sacc[r] - m_run);
                lsum += pv;
                if constexpr (DROP) {
                    const uint64_t off = (uint64_t)(8 * (r >> 2) + (r & 3)) * kLcgMul;
                    pv = lcg_keep(st_blk + off, thr) ? pv : 0.f;
                }
                pr[r] = pv;
            }
            l_run += lsum;
            // O^T += V^T P~^T: k-step r pairs lane-half h with key 8(r/4)+4h+r%4.
#pragma unroll
            for (int r = 0; r < 16; ++r) {
#pragma unroll
                for (int dt = 0; dt < DV / 32; ++dt) {
                    const float a = Vs[(8 * (r >> 2) + 4 * hh + (r & 3)) * VS + 32 * dt + l32];
                    oacc[dt] = mfma_f32(a, pr[r], oacc[dt]);
                }
            }
        }

        if (has_next) {
            float* Kn = lds + ((blk + 1) & 1) * Cfg::STAGE;
            kst.template store<KS>(Kn, tid);
            vst.template store<VS>(Kn + Cfg::KT, tid);
        }
        __syncthreads();
    }

    const float l_tot = xhalf_sum(l_run);
    if (my_q < S_q) {
        const float m_nat = (l_tot > 0.f) ? m_run * kLn2 : kNegInf;
        if (hh == 0) p.stats[(size_t)b * S_q + my_q] = m_nat + logf(l_tot + kEps);
        const float inv = (l_tot > kEps) ? p.c.keep_scale / l_tot : 0.f;
        float* Ob = static_cast<float*>(p.o) + ((size_t)b * S_q + my_q) * D_v;
#pragma unroll
        for (int dt = 0; dt < DV / 32; ++dt) {
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const int d0 = 32 * dt + 8 * g4 + 4 * hh;
                floatx4 fv;
#pragma unroll
                for (int e = 0; e < 4; ++e) fv[e] = oacc[dt][4 * g4 + e] * inv;
                if constexpr (VEC) {
                    if (d0 < D_v) *reinterpret_cast<floatx4*>(Ob + d0) = fv;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (d0 + e < D_v) Ob[d0 + e] = fv[e];
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// dK/dV at D <= 64: four waves, each all of its 32 keys (K, V, dK and dV fit
// in one wave's registers there).  Against the split roles below: B 16, S_q
// 512, S_kv 9000, D 32 256 -> 227 us, D 64 423 -> 398.
// ---------------------------------------------------------------------------
template <int DQK, int DV>
struct DkvWaveChainCfg {
    static constexpr int NT = 256, BKV = 128, BQ = 32;
    static constexpr int QS = DQK + 4, OS = DV + 4;
    static constexpr int QT = BQ * QS, OT = BQ * OS;
    static constexpr int STAGE = QT + OT + 2 * BQ;  // floats: Q, dO, stats2, delta
    static constexpr size_t LDS_BYTES = 2 * (size_t)STAGE * sizeof(float);
};

template <int DQK, int DV, bool VEC, bool DROP>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void sdpa_bwd_dkdv_f32_chain_wave_kernel(const BwdParams p) {
    using Cfg = DkvWaveChainCfg<DQK, DV>;
    constexpr int BKV = Cfg::BKV, BQ = Cfg::BQ, QS = Cfg::QS, OS = Cfg::OS;
    constexpr int HQ = DQK / 2, HV = DV / 2;
    float* lds = reinterpret_cast<float*>(smem);

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l32 = lane & 31, hh = lane >> 5;
    const int B = p.s.B, S_q = p.s.S_q, S_kv = p.s.S_kv, D_qk = p.s.D_qk, D_v = p.s.D_v;
    const bool causal = p.c.causal != 0;
    const int tiles = (S_kv + BKV - 1) / BKV;
    int b, kt;
    map_q_tile(blockIdx.x, B, tiles, false, b, kt);
    const int k0 = kt * BKV, kw0 = k0 + wave * 32, my_k = kw0 + l32;
    const bool key_ok = my_k < S_kv;

    const float* Qb = static_cast<const float*>(p.q) + (size_t)b * S_q * D_qk;
    const float* dOb = static_cast<const float*>(p.d_o) + (size_t)b * S_q * D_v;
    const float* Kb = static_cast<const float*>(p.k) + (size_t)b * S_kv * D_qk;
    const float* Vb = static_cast<const float*>(p.v) + (size_t)b * S_kv * D_v;
    const float* statsb = p.stats + (size_t)b * S_q;
    const float* deltab = p.delta + (size_t)b * S_q;

    float kf[HQ], vf[HV];
#pragma unroll
    for (int u = 0; u < HQ / 4; ++u) {
        const floatx4 f = __builtin_bit_cast(floatx4, load_row_chunk<float, VEC>(Kb, my_k, S_kv, HQ * hh + 4 * u, D_qk, D_qk));
#pragma unroll
        for (int e = 0; e < 4; ++e) kf[4 * u + e] = f[e];
    }
#pragma unroll
    for (int u = 0; u < HV / 4; ++u) {
        const floatx4 f = __builtin_bit_cast(floatx4, load_row_chunk<float, VEC>(Vb, my_k, S_kv, HV * hh + 4 * u, D_v, D_v));
#pragma unroll
        for (int e = 0; e < 4; ++e) vf[4 * u + e] = f[e];
    }
    prologue_loads_landed();

    const int q_begin = causal ? (min(k0, S_q) / BQ) * BQ : 0;
    const int nblk = (S_q - q_begin + BQ - 1) / BQ;
    const bool wave_live = kw0 < S_kv;
    const float sl2 = p.c.scale_log2;
    const float ksc = p.c.keep_scale;
    const uint64_t st_base = DROP ? lcg_state(p.c.seed_offset, (uint64_t)b * S_q + 4 * hh, (uint64_t)S_kv, my_k) : 0;
    const uint64_t row_step = (uint64_t)S_kv * kLcgMul;
    const uint32_t thr = p.c.drop_threshold;

    floatx16 dkacc[DQK / 32], dvacc[DV / 32];
#pragma unroll
    for (int dt = 0; dt < DQK / 32; ++dt) dkacc[dt] = floatx16{};
#pragma unroll
    for (int dt = 0; dt < DV / 32; ++dt) dvacc[dt] = floatx16{};

    TileStage<float, BQ, DQK, Cfg::NT, VEC> qst;
    TileStage<float, BQ, DV, Cfg::NT, VEC> ost;
    float fpre = 0.f;
    auto load_rows = [&](int q0) {
        qst.template load<false>(Qb, q0, S_q - q0, D_qk, D_qk, tid);
        ost.template load<false>(dOb, q0, S_q - q0, D_v, D_v, tid);
        if (tid < 2 * BQ) {
            const int r = q0 + (tid & (BQ - 1));
            if (tid < BQ) fpre = r < S_q ? statsb[r] * kLog2e : INFINITY;
            else fpre = r < S_q ? deltab[r] : 0.f;
        }
    };
    auto store_rows = [&](int s) {
        float* base = lds + s * Cfg::STAGE;
        qst.template store<QS>(base, tid);
        ost.template store<OS>(base + Cfg::QT, tid);
        if (tid < 2 * BQ) base[Cfg::QT + Cfg::OT + tid] = fpre;
    };

    if (nblk > 0) {
        load_rows(q_begin);
        store_rows(0);
    }
    __syncthreads();

    for (int blk = 0; blk < nblk; ++blk) {
        const int q0 = q_begin + blk * BQ;
        const int cur = blk & 1;
        const float* Qs = lds + cur * Cfg::STAGE;
        const float* dOs = Qs + Cfg::QT;
        const float* Fs = dOs + Cfg::OT;
        const bool has_next = blk + 1 < nblk;
        if (has_next) load_rows(q0 + BQ);

        if (wave_live && (!causal || q0 + BQ - 1 >= kw0)) {
            floatx16 sacc = floatx16{}, dpacc = floatx16{};
#pragma unroll
            for (int u = 0; u < HQ / 4; ++u) {
                const floatx4 qq = *reinterpret_cast<const floatx4*>(Qs + l32 * QS + HQ * hh + 4 * u);
#pragma unroll
                for (int e = 0; e < 4; ++e) sacc = mfma_f32(qq[e], kf[4 * u + e], sacc);
            }
#pragma unroll
            for (int u = 0; u < HV / 4; ++u) {
                const floatx4 oo = *reinterpret_cast<const floatx4*>(dOs + l32 * OS + HV * hh + 4 * u);
#pragma unroll
                for (int e = 0; e < 4; ++e) dpacc = mfma_f32(oo[e], vf[4 * u + e], dpacc);
            }
            const bool need_mask = !key_ok || (causal && q0 < kw0 + 31);
            const uint64_t st_blk = DROP ? st_base + (uint64_t)q0 * row_step : 0;
            float pk[16], ds[16];
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const int rb = 8 * g4 + 4 * hh;
                const floatx4 st4 = *reinterpret_cast<const floatx4*>(Fs + rb);
                const floatx4 de4 = *reinterpret_cast<const floatx4*>(Fs + BQ + rb);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int r = 4 * g4 + e;
                    float x = __builtin_fmaf(sacc[r], sl2, -st4[e]);
                    if (need_mask) {
                        const int q = q0 + rb + e;
                        if (!key_ok || (causal && my_k > q)) x = -INFINITY;
                    }
                    const float pr = fast_exp2(x);
                    const float p0 = pr > kEps ? pr : 0.f;
                    float dpk = DROP ? dpacc[r] * ksc : dpacc[r];
                    float pkk = p0;
                    if constexpr (DROP) {
                        const uint64_t off = (uint64_t)(8 * g4 + e) * row_step;
                        const bool keep = lcg_keep(st_blk + off, thr);
                        dpk = keep ? dpk : 0.f;
                        pkk = keep ? p0 : 0.f;
                    }
                    pk[r] = pkk;
                    ds[r] = p0 * (dpk - de4[e]);
                }
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int qrow = 8 * (r >> 2) + 4 * hh + (r & 3);
#pragma unroll
                for (int dt = 0; dt < DV / 32; ++dt)
                    dvacc[dt] = mfma_f32(dOs[qrow * OS + 32 * dt + l32], pk[r], dvacc[dt]);
#pragma unroll
                for (int dt = 0; dt < DQK / 32; ++dt)
                    dkacc[dt] = mfma_f32(Qs[qrow * QS + 32 * dt + l32], ds[r], dkacc[dt]);
            }
        }

        if (has_next) store_rows(cur ^ 1);
        __syncthreads();
    }

    if (key_ok) {
        const float sc = p.c.scale;
        float* dKb = static_cast<float*>(p.dk) + ((size_t)b * S_kv + my_k) * D_qk;
        float* dVb = static_cast<float*>(p.dv) + ((size_t)b * S_kv + my_k) * D_v;
#pragma unroll
        for (int dt = 0; dt < DQK / 32; ++dt)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const int d0 = 32 * dt + 8 * g4 + 4 * hh;
                floatx4 fv;
#pragma unroll
                for (int e = 0; e < 4; ++e) fv[e] = dkacc[dt][4 * g4 + e] * sc;
                if constexpr (VEC) {
                    if (d0 < D_qk) *reinterpret_cast<floatx4*>(dKb + d0) = fv;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (d0 + e < D_qk) dKb[d0 + e] = fv[e];
                }
            }
#pragma unroll
        for (int dt = 0; dt < DV / 32; ++dt)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const int d0 = 32 * dt + 8 * g4 + 4 * hh;
                floatx4 fv;
#pragma unroll
                for (int e = 0; e < 4; ++e) fv[e] = dvacc[dt][4 * g4 + e] * ksc;
                if constexpr (VEC) {
                    if (d0 < D_v) *reinterpret_cast<floatx4*>(dVb + d0) = fv;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (d0 + e < D_v) dVb[d0 + e] = fv[e];
                }
            }
    }
}

// ---------------------------------------------------------------------------
// dK/dV: two waves per group of 32 keys (P role: S, P~, dV; dS role: dP, dS,
// dK, one query block behind), blocks of 32 queries in a ring of three stages.
// ---------------------------------------------------------------------------
template <int DQK, int DV>
struct DkvChainCfg {
    static constexpr int NT = 512, BKV = 128, BQ = 32, NSTAGE = 3;
    static constexpr int QS = DQK + 4, OS = DV + 4;
    static constexpr int QT = BQ * QS, OT = BQ * OS;
    static constexpr int STAGE = QT + OT + 2 * BQ;  // floats: Q, dO, stats2, delta
    static constexpr int XB = 4 * 32 * 32;          // floats: P of 4 key groups x 32 queries
    static constexpr size_t LDS_BYTES = (NSTAGE * (size_t)STAGE + 2 * (size_t)XB) * sizeof(float);
    static_assert(LDS_BYTES <= 160 * 1024, "one workgroup per CU");
};

template <int DQK, int DV, bool VEC, bool DROP, bool DS>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void sdpa_bwd_dkdv_f32_chain_kernel(const BwdParams p) {
    using Cfg = DkvChainCfg<DQK, DV>;
    constexpr int BKV = Cfg::BKV, BQ = Cfg::BQ, QS = Cfg::QS, OS = Cfg::OS, NSTAGE = Cfg::NSTAGE;
    constexpr int HQ = DQK / 2, HV = DV / 2;
    float* lds = reinterpret_cast<float*>(smem);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kw = wave & 3;
    const int l32 = lane & 31, hh = lane >> 5;
    const int B = p.s.B, S_q = p.s.S_q, S_kv = p.s.S_kv, D_qk = p.s.D_qk, D_v = p.s.D_v;
    const bool causal = p.c.causal != 0;
    const int tiles = (S_kv + BKV - 1) / BKV;
    int b, kt;
    map_q_tile(blockIdx.x, B, tiles, false, b, kt);
    const int k0 = kt * BKV, kw0 = k0 + kw * 32, my_k = kw0 + l32;
    const bool key_ok = my_k < S_kv;

    const float* Qb = static_cast<const float*>(p.q) + (size_t)b * S_q * D_qk;
    const float* dOb = static_cast<const float*>(p.d_o) + (size_t)b * S_q * D_v;
    const float* statsb = p.stats + (size_t)b * S_q;
    const float* deltab = p.delta + (size_t)b * S_q;

    const int q_begin = causal ? (min(k0, S_q) / BQ) * BQ : 0;
    const int nblk = (S_q - q_begin + BQ - 1) / BQ;
    const bool wave_live = kw0 < S_kv;
    // Block m is skipped by both roles when the key group sees none of it.
    auto live = [&](int q0) { return wave_live && (!causal || q0 + BQ - 1 >= kw0); };
    const float sl2 = p.c.scale_log2;
    const float ksc = p.c.keep_scale;

    TileStage<float, BQ, DQK, Cfg::NT, VEC> qst;
    TileStage<float, BQ, DV, Cfg::NT, VEC> ost;
    float fpre = 0.f;
    auto load_rows = [&](int q0) {
        qst.load(Qb, q0, S_q - q0, D_qk, D_qk, tid);
        ost.load(dOb, q0, S_q - q0, D_v, D_v, tid);
        if (tid < 2 * BQ) {
            const int r = q0 + (tid & (BQ - 1));
            if (tid < BQ) fpre = r < S_q ? statsb[r] * kLog2e : INFINITY;
            else fpre = r < S_q ? deltab[r] : 0.f;
        }
    };
    auto store_rows = [&](int s) {
        float* base = lds + s * Cfg::STAGE;
        qst.template store<QS>(base, tid);
        ost.template store<OS>(base + Cfg::QT, tid);
        if (tid < 2 * BQ) base[Cfg::QT + Cfg::OT + tid] = fpre;
    };
    // P of block m for this key group: 16 floats per lane, lane-contiguous.
    auto xbuf = [&](int m) { return lds + NSTAGE * Cfg::STAGE + (m & 1) * Cfg::XB + kw * 1024; };

    if (nblk > 0) {
        load_rows(q_begin);
        store_rows(0);
    }

    if (wave < 4) {
        // ------------------------------------------------------------ P role
        const float* Kb = static_cast<const float*>(p.k) + (size_t)b * S_kv * D_qk;
        float kf[HQ];
#pragma unroll
        for (int u = 0; u < HQ / 4; ++u) {
            const floatx4 f = __builtin_bit_cast(floatx4, load_row_chunk<float, VEC>(Kb, my_k, S_kv, HQ * hh + 4 * u, D_qk, D_qk));
#pragma unroll
            for (int e = 0; e < 4; ++e) kf[4 * u + e] = f[e];
        }
        prologue_loads_landed();
        const uint64_t st_base = DROP ? lcg_state(p.c.seed_offset, (uint64_t)b * S_q + 4 * hh, (uint64_t)S_kv, my_k) : 0;
        const uint64_t row_step = (uint64_t)S_kv * kLcgMul;
        const uint32_t thr = p.c.drop_threshold;
        floatx16 dvacc[DV / 32];
#pragma unroll
        for (int dt = 0; dt < DV / 32; ++dt) dvacc[dt] = floatx16{};

        for (int n = 0; n <= nblk; ++n) {
            __syncthreads();
            const bool has_next = n + 1 < nblk;
            if (has_next) load_rows(q_begin + (n + 1) * BQ);
            const int q0 = q_begin + n * BQ;
            if (n < nblk && live(q0)) {
                const float* Qs = lds + (n % NSTAGE) * Cfg::STAGE;
                const float* dOs = Qs + Cfg::QT;
                const float* Fs = dOs + Cfg::OT;
                floatx16 sacc = floatx16{};
#pragma unroll
                for (int u = 0; u < HQ / 4; ++u) {
                    const floatx4 qq = *reinterpret_cast<const floatx4*>(Qs + l32 * QS + HQ * hh + 4 * u);
#pragma unroll
                    for (int e = 0; e < 4; ++e) sacc = mfma_f32(qq[e], kf[4 * u + e], sacc);
                }
                const bool need_mask = !key_ok || (causal && q0 < kw0 + 31);
                const uint64_t st_blk = DROP ? st_base + (uint64_t)q0 * row_step : 0;
                float* xs = xbuf(n);
#pragma unroll
                for (int g4 = 0; g4 < 4; ++g4) {
                    const int rb = 8 * g4 + 4 * hh;
                    const floatx4 st4 = *reinterpret_cast<const floatx4*>(Fs + rb);
                    floatx4 xv;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int r = 4 * g4 + e;
                        float x = __builtin_fmaf(sacc[r], sl2, -st4[e]);
                        if (need_mask) {
                            const int q = q0 + rb + e;
                            if (!key_ok || (causal && my_k > q)) x = -INFINITY;
                        }
                        const float pr = fast_exp2(x);
                        const float p0 = pr > kEps ? pr : 0.f;
                        float pkk = p0;
                        if constexpr (DROP) {
                            const bool keep = lcg_keep(st_blk + (uint64_t)(8 * g4 + e) * row_step, thr);
                            pkk = keep ? p0 : 0.f;
                            xv[e] = keep ? p0 : -p0;
                        } else {
                            xv[e] = p0;
                        }
                        sacc[r] = pkk;
                    }
                    *reinterpret_cast<floatx4*>(xs + (g4 * 64 + lane) * 4) = xv;
                }
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int qrow = 8 * (r >> 2) + 4 * hh + (r & 3);
#pragma unroll
                    for (int dt = 0; dt < DV / 32; ++dt)
                        dvacc[dt] = mfma_f32(dOs[qrow * OS + 32 * dt + l32], sacc[r], dvacc[dt]);
                }
            }
            if (has_next) store_rows((n + 1) % NSTAGE);
        }
        if (key_ok) {
            float* dVb = static_cast<float*>(p.dv) + ((size_t)b * S_kv + my_k) * D_v;
#pragma unroll
            for (int dt = 0; dt < DV / 32; ++dt)
#pragma unroll
                for (int g4 = 0; g4 < 4; ++g4) {
                    const int d0 = 32 * dt + 8 * g4 + 4 * hh;
                    floatx4 fv;
#pragma unroll
                    for (int e = 0; e < 4; ++e) fv[e] = dvacc[dt][4 * g4 + e] * ksc;
                    if constexpr (VEC) {
                        if (d0 < D_v) *reinterpret_cast<floatx4*>(dVb + d0) = fv;
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (d0 + e < D_v) dVb[d0 + e] = fv[e];
                    }
                }
        }
    } else {
        // ----------------------------------------------------------- dS role
        const float* Vb = static_cast<const float*>(p.v) + (size_t)b * S_kv * D_v;
        float vf[HV];
#pragma unroll
        for (int u = 0; u < HV / 4; ++u) {
            const floatx4 f = __builtin_bit_cast(floatx4, load_row_chunk<float, VEC>(Vb, my_k, S_kv, HV * hh + 4 * u, D_v, D_v));
#pragma unroll
            for (int e = 0; e < 4; ++e) vf[4 * u + e] = f[e];
        }
        prologue_loads_landed();
        floatx16 dkacc[DQK / 32];
#pragma unroll
        for (int dt = 0; dt < DQK / 32; ++dt) dkacc[dt] = floatx16{};
        // dS path: this key group's dS of each visited block goes to its
        // chunk (DsLayout32): the lane's 16 values, query positions 16 hh + r,
        // as four 16-byte slots, one per store, each store 1 KB whole; zero
        // for keys past S_kv (the dQ kernel reads them unmasked)
        const DsLayout32 dsl(S_q, S_kv, causal);

        for (int n = 0; n <= nblk; ++n) {
            __syncthreads();
            const bool has_next = n + 1 < nblk;
            if (has_next) load_rows(q_begin + (n + 1) * BQ);
            const int m = n - 1;
            const int q0 = q_begin + m * BQ;
            if (m >= 0 && live(q0)) {
                const float* Qs = lds + (m % NSTAGE) * Cfg::STAGE;
                const float* dOs = Qs + Cfg::QT;
                const float* Fs = dOs + Cfg::OT;
                floatx16 dpacc = floatx16{};
#pragma unroll
                for (int u = 0; u < HV / 4; ++u) {
                    const floatx4 oo = *reinterpret_cast<const floatx4*>(dOs + l32 * OS + HV * hh + 4 * u);
#pragma unroll
                    for (int e = 0; e < 4; ++e) dpacc = mfma_f32(oo[e], vf[4 * u + e], dpacc);
                }
                // dS = P0 (keep ? dP / (1-p) : 0 - delta), P0 = |x|, keep = x > 0
                const float* xs = xbuf(m);
#pragma unroll
                for (int g4 = 0; g4 < 4; ++g4) {
                    const floatx4 xv = *reinterpret_cast<const floatx4*>(xs + (g4 * 64 + lane) * 4);
                    const floatx4 de4 = *reinterpret_cast<const floatx4*>(Fs + BQ + 8 * g4 + 4 * hh);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int r = 4 * g4 + e;
                        float dpk = DROP ? dpacc[r] * ksc : dpacc[r];
                        float p0 = xv[e];
                        if constexpr (DROP) {
                            dpk = xv[e] > 0.f ? dpk : 0.f;
                            p0 = __builtin_fabsf(xv[e]);
                        }
                        dpacc[r] = p0 * (dpk - de4[e]);
                    }
                }
                if constexpr (DS) {
                    unsigned char* grp = static_cast<unsigned char*>(p.ds) + dsl.offset(b, kt, q0 / BQ) + kw * 4096;
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        floatx4 v;
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = key_ok ? dpacc[4 * u + e] : 0.f;
                        __builtin_nontemporal_store(
                            v, reinterpret_cast<floatx4*>(grp + DsLayout32::slot32(l32, 16 * hh + 4 * u)));
                    }
                }
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int qrow = 8 * (r >> 2) + 4 * hh + (r & 3);
#pragma unroll
                    for (int dt = 0; dt < DQK / 32; ++dt)
                        dkacc[dt] = mfma_f32(Qs[qrow * QS + 32 * dt + l32], dpacc[r], dkacc[dt]);
                }
            }
            if (has_next) store_rows((n + 1) % NSTAGE);
        }
        if (key_ok) {
            const float sc = p.c.scale;
            float* dKb = static_cast<float*>(p.dk) + ((size_t)b * S_kv + my_k) * D_qk;
#pragma unroll
            for (int dt = 0; dt < DQK / 32; ++dt)
#pragma unroll
                for (int g4 = 0; g4 < 4; ++g4) {
                    const int d0 = 32 * dt + 8 * g4 + 4 * hh;
                    floatx4 fv;
#pragma unroll
                    for (int e = 0; e < 4; ++e) fv[e] = dkacc[dt][4 * g4 + e] * sc;
                    if constexpr (VEC) {
                        if (d0 < D_qk) *reinterpret_cast<floatx4*>(dKb + d0) = fv;
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (d0 + e < D_qk) dKb[d0 + e] = fv[e];
                    }
                }
        }
    }
}

}  // namespace

hipError_t launch_fwd_f32_chain(const FwdParams& p, bool vec, hipStream_t stream) {
    return with_dim(p.s.D_qk, [&](auto dqk) {
        return with_dim(p.s.D_v, [&](auto dv) {
            return with_bool(vec, [&](auto v) {
                return with_bool(p.c.use_dropout != 0, [&](auto d) {
                    constexpr int DQK = decltype(dqk)::value, DV = decltype(dv)::value;
                    using Cfg = FwdChainCfg<DQK, DV>;
                    const unsigned n = (unsigned)((p.s.S_q + Cfg::BM - 1) / Cfg::BM * p.s.B);
                    return launch_kernel<sdpa_fwd_f32_chain_kernel<DQK, DV, decltype(v)::value, decltype(d)::value>>(
                        n, Cfg::NT, Cfg::LDS_BYTES, stream, p);
                });
            });
        });
    });
}

hipError_t launch_bwd_dkdv_f32_chain(const BwdParams& p, bool vec, hipStream_t stream) {
    return with_dim(p.s.D_qk, [&](auto dqk) {
        return with_dim(p.s.D_v, [&](auto dv) {
            return with_bool(vec, [&](auto v) {
                return with_bool(p.c.use_dropout != 0, [&](auto d) {
                    constexpr int DQK = decltype(dqk)::value, DV = decltype(dv)::value;
                    constexpr bool V = decltype(v)::value, D = decltype(d)::value;
                    using Cfg = DkvChainCfg<DQK, DV>;
                    static_assert(Cfg::BKV == DsLayout32::KT && Cfg::BQ == DsLayout32::QBK, "dS chunk geometry");
                    const unsigned n = (unsigned)((p.s.S_kv + Cfg::BKV - 1) / Cfg::BKV * p.s.B);
                    if constexpr (V && (DQK == 128 || DV == 128)) {
                        if (p.ds)
                            return launch_kernel<sdpa_bwd_dkdv_f32_chain_kernel<DQK, DV, V, D, true>>(n, Cfg::NT, Cfg::LDS_BYTES,
                                                                                                 stream, p);
                    }
                    if (p.ds) return hipErrorInvalidValue;
                    if constexpr (DQK == 128 || DV == 128) {
                        return launch_kernel<sdpa_bwd_dkdv_f32_chain_kernel<DQK, DV, V, D, false>>(n, Cfg::NT, Cfg::LDS_BYTES,
                                                                                              stream, p);
                    } else {
                        using CW = DkvWaveChainCfg<DQK, DV>;
                        static_assert(CW::BKV == Cfg::BKV, "same grid");
                        return launch_kernel<sdpa_bwd_dkdv_f32_chain_wave_kernel<DQK, DV, V, D>>(n, CW::NT, CW::LDS_BYTES,
                                                                                            stream, p);
                    }
                });
            });
        });
    });
}

}  // namespace sdpa
