// sdpa_f16_fwd_small.hip -- fp16 Sdpa forward for gfx950 where the query side
// has too few tiles to fill the chip: token generation, a few queries against
// a long memory, short sequences, few heads.
//
// The kernel of sdpa_f16_fwd.hip gives a workgroup 128 queries and all of
// their keys; with few such tiles most of the 256 CUs idle, and each busy one
// runs a long serial chain of key blocks.  Here a workgroup owns 32 queries,
// its four waves take the 32-key blocks in turn, each wave with running
// statistics and an accumulator of its own (merged through LDS at the end),
// and the blocks of one tile may further be divided over several workgroups
// (sdpa_parts.h), whose results a second kernel merges from the caller's workspace.
//
// Each wave streams its own K/V blocks through a two-stage LDS ring (the
// copies of sdpa_dma.h): no two waves share a block, so the loop has no
// barrier, only waits on the wave's own copies.  The price is that the K/V
// rows go to LDS once per 32 queries instead of once per 128.
//
// Element semantics are those of sdpa_f16_fwd.hip (hi/lo split of P~
// included; its test sees the mass of this wave's earlier keys only, which
// errs towards splitting).
#include "sdpa_launch.h"
#include "sdpa_merge.h"
#include "sdpa_params.h"
#include "sdpa_parts.h"
#include "sdpa_wave.h"

namespace sdpa {
namespace {

constexpr float kTauW = 8.0f;  // lazy-rescale threshold (log2 units), as in sdpa_f16_fwd.hip

template <int DQK, int DV>
struct FwdWaveCfg {
    static constexpr int NW = 4, NT = 64 * NW, BM = 32, BN = 32;
    static constexpr int LK = DQK / 8, LV = DV / 8;
    static constexpr int KB = BN * DQK * 2, VB = BN * DV * 2, STAGE = KB + VB, RING = 2 * STAGE;
    // merge area (after the loop): O of every wave, then m and l
    static constexpr int OS = acc_stride(DV), MERGE = NW * BM * OS * 4 + NW * BM * 8;
    static constexpr size_t LDS_BYTES = NW * RING > MERGE ? NW * RING : MERGE;
    static_assert(LDS_BYTES <= 160 * 1024, "gfx950 LDS");
    static constexpr int WPE = 2 * LDS_BYTES <= 160 * 1024 ? 2 : 1;
    static constexpr int COPIES = WaveCopy<LK, false>::LOADS + WaveCopy<LV, true>::LOADS;
    static_assert(COPIES < 64, "vmcnt is 6 bits");
};

template <int DQK, int DV, bool CAUSAL, bool DROP, bool P4>
__global__ __launch_bounds__((FwdWaveCfg<DQK, DV>::NT))
__attribute__((amdgpu_waves_per_eu(FwdWaveCfg<DQK, DV>::WPE, FwdWaveCfg<DQK, DV>::WPE)))
void sdpa_fwd_f16_wave_kernel(const FwdParams p, const int win) {
    using Cfg = FwdWaveCfg<DQK, DV>;
    constexpr int BM = Cfg::BM, BN = Cfg::BN, LK = Cfg::LK, LV = Cfg::LV, NW = Cfg::NW;
    constexpr int NKS = DQK / 16, NDT = DV / 32;

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int B = p.s.B, S_q = p.s.S_q, S_kv = p.s.S_kv, D_qk = p.s.D_qk, D_v = p.s.D_v;
    const int np = p.parts, items = (S_q + BM - 1) / BM * np;
    int b, it;
    xcd_map(blockIdx.x, B * items, items, CAUSAL, win, b, it);
    const int qt = it / np, part = it - qt * np;
    const int q0 = qt * BM, my_q = q0 + l32;

    const half_t* Qb = static_cast<const half_t*>(p.q) + (size_t)b * S_q * D_qk;
    const RowSrc ksrc = row_src(p.k, (size_t)b * S_kv, S_kv, D_qk * 2);
    const RowSrc vsrc = row_src(p.v, (size_t)b * S_kv, S_kv, D_v * 2);

    // |scale| with negated queries for scale < 0; 1e-30 for 0 (sdpa_f16_fwd.hip)
    const float sl2_raw = p.c.scale_log2;
    const bool neg = sl2_raw < 0.f;
    const float sl2 = (sl2_raw == 0.f) ? 1e-30f : fabsf(sl2_raw);

    // this wave's blocks: lo + wave, lo + wave + NW, ... below hi
    const int nblk = (min(S_kv, CAUSAL ? q0 + BM : S_kv) + BN - 1) / BN;
    const int lo = part_begin(nblk, part, np), hi = part_begin(nblk, part + 1, np);
    const uint32_t ring = lds_base() + (uint32_t)(wave * Cfg::RING);
    WaveCopy<LK, false> kc;
    WaveCopy<LV, true> vc;
    kc.init(lane, D_qk * 2, (D_qk + 7) / 8);
    vc.init(lane, D_v * 2, (D_v + 7) / 8);
    auto issue = [&](int blk, uint32_t so) {
        kc.issue(ksrc.shifted(blk * BN), ring + so);
        vc.issue(vsrc.shifted(blk * BN), ring + so + (uint32_t)Cfg::KB);
    };
    half8 qreg[NKS];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
        half8 v = __builtin_bit_cast(half8, load_row_chunk<half_t, !P4>(Qb, my_q, S_q, 16 * ks + 8 * hh, D_qk, D_qk));
        qreg[ks] = neg ? -v : v;
    }
    prologue_loads_landed();
    if (lo + wave < hi) issue(lo + wave, 0);

    SwzLane<LK> swK;
    swK.init(lane);
    const uint32_t rkl = ring + swK.row;                          // K rows (^ 32 ks)
    const uint32_t tvl = ring + Cfg::KB + tr_lane_off<LV>(lane);  // V^T (^ 64 dt)

    floatx16 oacc[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) oacc[dt] = floatx16{};
    float m_run = kMaxSentinel, l_run = 0.f;
    // hash of (my_q, key 4 hh of the wave's current block)
    uint64_t st = DROP ? lcg_state(p.c.seed_offset, (uint64_t)b * S_q + my_q, (uint64_t)S_kv,
                                   (uint64_t)((lo + wave) * BN + 4 * hh))
                       : 0;
    const uint32_t thr = p.c.drop_threshold;

    uint32_t so = 0;
    for (int blk = lo + wave; blk < hi; blk += NW, so ^= (uint32_t)Cfg::STAGE) {
        // the other stage's block has been read; the next block's copies go
        // out there, and this block's have landed once only those are in flight
        lds_reads_done();
        if (blk + NW < hi) {
            issue(blk + NW, so ^ (uint32_t)Cfg::STAGE);
            wait_copies<Cfg::COPIES>();
        } else {
            wait_copies<0>();
        }
        const int kv0 = blk * BN;
        const float split_thr = m_run + fast_log2(xhalf_sum(l_run)) + kSplitLog2;
        floatx16 s = floatx16{};
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) s = mfma_f16(keep4<P4>(ld_b128((rkl ^ (uint32_t)(32 * ks)) + so), ks, hh, D_qk), qreg[ks], s);
        half8 av[2][NDT];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) {
                const uint32_t a = (tvl ^ (uint32_t)(64 * dt)) + so + 16 * LV * 16 * j;
                av[j][dt] = ld_tr8(a, a + 16 * LV * 8);
            }
        if (kv0 + BN > S_kv || (CAUSAL && kv0 + BN - 1 > q0)) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int key = kv0 + 8 * (r >> 2) + 4 * hh + (r & 3);
                if (key >= S_kv || (CAUSAL && key > my_q)) s[r] = -INFINITY;
            }
        }
        float mx = s[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
        mx = xhalf_max(mx) * sl2;
        const float m_use = (mx > m_run + kTauW) ? fmaxf(m_run, mx) : m_run;
        const float alpha = fast_exp2(m_run - m_use);
        float lq[4];
        float pf[16];
        uint64_t sg = st;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
#pragma unroll
            for (int e = 0; e < 4; ++e) pf[4 * g + e] = fast_exp2(__builtin_fmaf(s[4 * g + e], sl2, -m_use));
            lq[g] = (pf[4 * g] + pf[4 * g + 1]) + (pf[4 * g + 2] + pf[4 * g + 3]);
            if constexpr (DROP) {
                uint64_t se = sg;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    pf[4 * g + e] = lcg_keep(se, thr) ? pf[4 * g + e] : 0.f;
                    se += kLcgMul;
                }
                sg += 8 * kLcgMul;
            }
        }
        if constexpr (DROP) st += (uint64_t)(NW * BN) * kLcgMul;
        if (wave_any(alpha != 1.f)) {
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) oacc[dt][r] *= alpha;
        }
        l_run = __builtin_fmaf(l_run, alpha, (lq[0] + lq[1]) + (lq[2] + lq[3]));
        m_run = m_use;
        half8 pb[2];
#pragma unroll
        for (int j = 0; j < 2; ++j)
            pb[j] = half8_of(pack_h2(pf[8 * j], pf[8 * j + 1]), pack_h2(pf[8 * j + 2], pf[8 * j + 3]),
                             pack_h2(pf[8 * j + 4], pf[8 * j + 5]), pack_h2(pf[8 * j + 6], pf[8 * j + 7]));
        if (wave_any(mx > split_thr)) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                float lo8[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) lo8[i] = pf[8 * j + i] - (float)pb[j][i];
                const half8 pl = half8_of(pack_h2(lo8[0], lo8[1]), pack_h2(lo8[2], lo8[3]),
                                          pack_h2(lo8[4], lo8[5]), pack_h2(lo8[6], lo8[7]));
#pragma unroll
                for (int dt = 0; dt < NDT; ++dt) oacc[dt] = mfma_f16(av[j][dt], pl, oacc[dt]);
            }
        }
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) oacc[dt] = mfma_f16(av[j][dt], pb[j], oacc[dt]);
    }

    // ---- merge the four waves: every ring has been read
    const float l_tot = xhalf_sum(l_run);
    __syncthreads();
    float* mo = reinterpret_cast<float*>(smem);
    float* mml = mo + NW * BM * Cfg::OS;
    if (hh == 0) {
        mml[(wave * BM + l32) * 2] = m_run;
        mml[(wave * BM + l32) * 2 + 1] = l_tot;
    }
    acc_to_lds<DV>(mo, wave * BM + l32, oacc, hh);
    __syncthreads();
    // one thread per four columns of a row
    const bool whole = np == 1;
#pragma unroll
    for (int i0 = 0; i0 < BM * (DV / 4); i0 += Cfg::NT) {
        const int i = i0 + tid, row = i / (DV / 4), c = 4 * (i % (DV / 4)), q = q0 + row;
        if ((BM * (DV / 4) % Cfg::NT && i >= BM * (DV / 4)) || q >= S_q || c >= D_v) continue;
        float mw[NW], lw[NW], M = kMaxSentinel;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            mw[w] = mml[(w * BM + row) * 2];
            lw[w] = mml[(w * BM + row) * 2 + 1];
            M = fmaxf(M, mw[w]);
        }
        float L = 0.f;
        floatx4 acc = floatx4{};
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float f = fast_exp2(mw[w] - M);
            L = __builtin_fmaf(lw[w], f, L);
            const floatx4 x = *reinterpret_cast<const floatx4*>(mo + (w * BM + row) * Cfg::OS + c);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] = __builtin_fmaf(x[e], f, acc[e]);
        }
        const size_t grow = (size_t)b * S_q + q;
        if (whole) {
            if (c == 0) p.stats[grow] = ((L > 0.f) ? M * kLn2 : kNegInf) + logf(L + kEps);
            const float inv = (L > kEps) ? p.c.keep_scale / L : 0.f;
            *reinterpret_cast<half4*>(static_cast<half_t*>(p.o) + grow * D_v + c) = scaled_h4(acc, inv);
        } else {
            const size_t at = (size_t)part * B * S_q + grow;
            if (c == 0) {
                p.part_ml[2 * at] = M;
                p.part_ml[2 * at + 1] = L;
            }
            *reinterpret_cast<floatx4*>(p.part_o + at * D_v + c) = acc;
        }
    }
}

}  // namespace

hipError_t launch_fwd_f16_wave(const FwdParams& p, hipStream_t stream) {
    const int B = p.s.B, S_q = p.s.S_q;
    if (B == 0 || S_q == 0) return hipSuccess;
    return with_dim(p.s.D_qk, [&](auto dqk) {
        return with_dim(p.s.D_v, [&](auto dv) {
            return with_bool(p.c.causal != 0, [&](auto c) {
                return with_bool(p.c.use_dropout != 0, [&](auto d) {
                    constexpr int DQK = decltype(dqk)::value, DV = decltype(dv)::value;
                    using Cfg = FwdWaveCfg<DQK, DV>;
                    static_assert(Cfg::BM == kSmallRows && Cfg::BN == kSmallRows && Cfg::NW == kSmallWaves, "planned by fwd_plan");
                    const long long n = (long long)((S_q + Cfg::BM - 1) / Cfg::BM) * p.parts * B;
                    constexpr bool CA = decltype(c)::value, DR = decltype(d)::value;
                    const int win = row_window((size_t)p.s.S_kv * (DQK + DV) * 2);
                    hipError_t err = hipErrorInvalidValue;
                    if (p.s.D_qk % 8 == 0 && p.s.D_v % 8 == 0)
                        err = launch_kernel<sdpa_fwd_f16_wave_kernel<DQK, DV, CA, DR, false>>((unsigned)n, Cfg::NT, Cfg::LDS_BYTES,
                                                                                          stream, p, win);
                    else if constexpr (DQK <= 64 && DV <= 64)
                        err = launch_kernel<sdpa_fwd_f16_wave_kernel<DQK, DV, CA, DR, true>>((unsigned)n, Cfg::NT, Cfg::LDS_BYTES,
                                                                                         stream, p, win);
                    return err == hipSuccess && p.parts > 1 ? launch_fwd_merge<half_t>(p, stream) : err;
                });
            });
        });
    });
}

}  // namespace sdpa
