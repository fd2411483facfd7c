// sdpa_f16_bwd_small.hip -- fp16 SdpaGrad kernels for gfx950 where a side has
// too few tiles to fill the chip (few batch rows, short sequences, a few
// queries against a long memory).
//
// The kernels of sdpa_f16_dq/dkdv*.hip give a workgroup 128 queries (256 for
// dQ from dS) or 128 keys and the whole other side; with few such tiles most
// of the 256 CUs idle and the busy ones each run a long serial chain.  Here a
// workgroup owns 32 queries (64 for dQ from dS) or 32 keys, its four waves
// take the 32-row blocks of the other side in turn, each streaming them
// through an LDS ring of its own (sdpa_wave.h; no barrier in the loop), and
// their accumulators are summed through LDS, in wave order, at the end.  The
// dQ kernel may further divide a tile's keys over workgroups, whose sums a
// second kernel adds in part order from the caller's workspace.
//
// D <= 64 may also be a multiple of 4 only (P4, keep4), which the large
// kernels' copies do not take: the register-staged kernels served such shapes
// (step of B 20, S 400, D 32/4, dropout: 87 -> 33 us).
//
// Element semantics are those of the large kernels (sdpa_bwd.hip restates the
// reference's, sdpa/sdpa_bwd.cu.cc:130-170, 291-327).
#include <type_traits>

#include "sdpa_launch.h"
#include "sdpa_params.h"
#include "sdpa_parts.h"
#include "sdpa_wave.h"

namespace sdpa {
namespace {

// P of a score x = s scale log2(e) - stats log2(e), 0 where P <= 1e-6.  P4
// compares, as the register-staged kernels of these shapes do; the other
// shapes have kGateShift in x, as their large kernels do (in bits of x that
// lie below the rounding of P to fp16).  kGateScale enters here and not the
// factor that P meets: dP / (1-p) - delta times 2^106 passes the fp32 range
// at 4e6, and a weight of 0 would make NaN of it.
template <bool P4>
__device__ __forceinline__ float gated(float x) {
    const float pr = fast_exp2(x);
    if constexpr (P4) return pr > kEps ? pr : 0.f;
    return pr * kGateScale;
}

// ---------------------------------------------------------------------------
// dQ of 32 queries (D <= 64), with the row values for the dK/dV kernel
// ---------------------------------------------------------------------------
template <int DQK, int DV>
struct DqWaveCfg {
    static constexpr int NW = kSmallWaves, NT = 64 * NW, BM = kSmallRows, BN = 32;
    static constexpr int LK = DQK / 8, LV = DV / 8;
    static constexpr int KB = BN * DQK * 2, VB = BN * DV * 2, STAGE = KB + VB, RING = 2 * STAGE;
    static constexpr int MERGE = NW * BM * acc_stride(DQK) * 4;
    static constexpr size_t LDS_BYTES = NW * RING > MERGE ? NW * RING : MERGE;
    static_assert(2 * LDS_BYTES <= 160 * 1024, "two workgroups per CU");
    static constexpr int COPIES = WaveCopy<LK, false>::LOADS + WaveCopy<LV, false>::LOADS;
};

template <int DQK, int DV, bool CAUSAL, bool DROP, bool P4>
__global__ __launch_bounds__((DqWaveCfg<DQK, DV>::NT)) __attribute__((amdgpu_waves_per_eu(2, 2)))
void sdpa_bwd_dq_f16_wave_kernel(const BwdParams p, const int win) {
    using Cfg = DqWaveCfg<DQK, DV>;
    constexpr int BM = Cfg::BM, BN = Cfg::BN, LK = Cfg::LK, LV = Cfg::LV, NW = Cfg::NW;
    constexpr int NK = DQK / 16, NV = DV / 16, NDT = DQK / 32;

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int B = p.s.B, S_q = p.s.S_q, S_kv = p.s.S_kv, D_qk = p.s.D_qk, D_v = p.s.D_v;
    const int np = p.parts, items = (S_q + BM - 1) / BM * np;
    int b, it;
    xcd_map(blockIdx.x, B * items, items, CAUSAL, win, b, it);
    const int qt = it / np, part = it - qt * np;
    const int q0 = qt * BM, my_q = q0 + l32;
    const size_t row_q = (size_t)b * S_q + my_q;

    const half_t* Qb = static_cast<const half_t*>(p.q) + (size_t)b * S_q * D_qk;
    const half_t* Ob = static_cast<const half_t*>(p.o) + (size_t)b * S_q * D_v;
    const half_t* dOb = static_cast<const half_t*>(p.d_o) + (size_t)b * S_q * D_v;
    const RowSrc ksrc = row_src(p.k, (size_t)b * S_kv, S_kv, D_qk * 2);
    const RowSrc vsrc = row_src(p.v, (size_t)b * S_kv, S_kv, D_v * 2);

    const int nblk = (min(S_kv, CAUSAL ? q0 + BM : S_kv) + BN - 1) / BN;
    const int lo = part_begin(nblk, part, np), hi = part_begin(nblk, part + 1, np);
    const uint32_t ringo = (uint32_t)(wave * Cfg::RING), ring = lds_base() + ringo;
    WaveCopy<LK, false> kc;
    WaveCopy<LV, false> vc;
    kc.init(lane, D_qk * 2, (D_qk + 7) / 8);
    vc.init(lane, D_v * 2, (D_v + 7) / 8);
    auto issue = [&](int blk, uint32_t so) {
        kc.issue(ksrc.shifted(blk * BN), ring + so);
        vc.issue(vsrc.shifted(blk * BN), ring + so + (uint32_t)Cfg::KB);
    };

    // rows, delta and stats2 as the 128-query kernel forms them (same order)
    half8 qreg[NK], doreg[NV];
#pragma unroll
    for (int ks = 0; ks < NK; ++ks)
        qreg[ks] = __builtin_bit_cast(half8, load_row_chunk<half_t, !P4>(Qb, my_q, S_q, 16 * ks + 8 * hh, D_qk, D_qk));
    float dpart = 0.f;
#pragma unroll
    for (int ks = 0; ks < NV; ++ks) {
        doreg[ks] = __builtin_bit_cast(half8, load_row_chunk<half_t, !P4>(dOb, my_q, S_q, 16 * ks + 8 * hh, D_v, D_v));
        const half8 o8 = __builtin_bit_cast(half8, load_row_chunk<half_t, !P4>(Ob, my_q, S_q, 16 * ks + 8 * hh, D_v, D_v));
#pragma unroll
        for (int e = 0; e < 8; ++e) dpart += (float)doreg[ks][e] * (float)o8[e];
    }
    const float delta = xhalf_sum(dpart);
    const bool row_ok = my_q < S_q;
    const float stats = row_ok ? p.stats[row_q] : INFINITY;
    if (row_ok && hh == 0 && wave == 0 && part == 0) {
        p.delta[row_q] = delta;
        p.stats2[row_q] = __builtin_fmaf(stats, kLog2e, kGateShift);
    }
    prologue_loads_landed();
    if (lo + wave < hi) issue(lo + wave, 0);
    const float sl2 = p.c.scale_log2, ksc = p.c.keep_scale;
    const float nst = P4 ? -(stats * kLog2e) : -__builtin_fmaf(stats, kLog2e, kGateShift);

    uint64_t st = DROP ? lcg_state(p.c.seed_offset, row_q, (uint64_t)S_kv, (uint64_t)((lo + wave) * BN + 4 * hh)) : 0;
    const uint32_t thr = p.c.drop_threshold;
    SwzLane<LK> swK;
    SwzLane<LV> swV;
    swK.init(lane);
    swV.init(lane);
    floatx16 acc[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) acc[dt] = floatx16{};

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
        const int k0 = blk * BN;
        const uint32_t kb = ringo + so, vb = kb + (uint32_t)Cfg::KB;
        floatx16 s = floatx16{}, dp = floatx16{};
#pragma unroll
        for (int ks = 0; ks < NK; ++ks) s = mfma_f16(keep4<P4>(lds_row<LK>(kb + swK.row, ks, 0), ks, hh, D_qk), qreg[ks], s);
#pragma unroll
        for (int ks = 0; ks < NV; ++ks) dp = mfma_f16(keep4<P4>(lds_row<LV>(vb + swV.row, ks, 0), ks, hh, D_v), doreg[ks], dp);
        half8 at[2][NDT];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) at[j][dt] = lds_tr<LK>(kb + swK.tr0, kb + swK.tr1, dt, 16 * j);
        const bool mask = k0 + BN > S_kv || (CAUSAL && k0 + BN - 1 > q0);
        uint32_t w[8];
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
            float ds2[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int rr = r + e;
                float x = __builtin_fmaf(s[rr], sl2, nst);
                if (mask) {
                    const int key = k0 + 8 * (rr >> 2) + 4 * hh + (rr & 3);
                    if (key >= S_kv || (CAUSAL && key > my_q)) x = -INFINITY;
                }
                const float pr = gated<P4>(x);
                float t = __builtin_fmaf(dp[rr], ksc, -delta);
                if constexpr (DROP)
                    t = lcg_keep(st + (uint64_t)(8 * (rr >> 2) + (rr & 3)) * kLcgMul, thr) ? t : -delta;
                ds2[e] = pr * t;
            }
            w[r >> 1] = pack_h2(ds2[0], ds2[1]);
        }
        if constexpr (DROP) st += (uint64_t)(NW * BN) * kLcgMul;
        const half8 ds0 = half8_of(w[0], w[1], w[2], w[3]), ds1 = half8_of(w[4], w[5], w[6], w[7]);
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
            acc[dt] = mfma_f16(at[0][dt], ds0, acc[dt]);
            acc[dt] = mfma_f16(at[1][dt], ds1, acc[dt]);
        }
    }

    __syncthreads();  // every ring has been read
    float* m = reinterpret_cast<float*>(smem);
    acc_to_lds<DQK>(m, wave * BM + l32, acc, hh);
    __syncthreads();
    const size_t grow0 = (size_t)b * S_q + q0;
    sum_waves<NW, BM, DQK>(m, tid, S_q - q0, D_qk, [&](int row, int c, const floatx4& sum) {
        if (np == 1)
            *reinterpret_cast<half4*>(static_cast<half_t*>(p.dq) + (grow0 + row) * D_qk + c) = scaled_h4(sum, p.c.scale);
        else
            *reinterpret_cast<floatx4*>(p.part_dq + ((size_t)part * B * S_q + grow0 + row) * D_qk + c) = sum;
    });
}

// dQ of a row from its parts, added in part order.  One thread per four columns.
__global__ __launch_bounds__(256) void sdpa_bwd_dq_merge_f16_kernel(const BwdParams p) {
    const int cpr = p.s.D_qk / 4, np = p.parts;
    const size_t n = (size_t)p.s.B * p.s.S_q * cpr, i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const floatx4* src = reinterpret_cast<const floatx4*>(p.part_dq) + i;
    constexpr int U = 4;  // loads in flight before the first is used
    floatx4 s = floatx4{};
    for (int k0 = 0; k0 < np; k0 += U) {
        floatx4 x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) x[u] = src[(size_t)(k0 + u < np ? k0 + u : np - 1) * n];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (k0 + u < np) s += x[u];
    }
    *(reinterpret_cast<half4*>(p.dq) + i) = scaled_h4(s, p.c.scale);
}

// ---------------------------------------------------------------------------
// dK and dV of 32 keys; DS also stores dS' for the dS path (DsLayout)
// ---------------------------------------------------------------------------
template <int DQK, int DV>
struct DkvWaveCfg {
    static constexpr int NW = kSmallWaves, NT = 64 * NW, BKV = kSmallRows, BQ = 32;
    static constexpr int LQ = DQK / 8, LO = DV / 8;
    static constexpr int QB = BQ * DQK * 2, OB = BQ * DV * 2, FB = 2 * 256;  // stats (P4) or stats2, and delta: 64 floats each, 32 used
    static constexpr int STAGE = QB + OB + FB, RING = 2 * STAGE;
    static constexpr int MERGE = NW * BKV * (acc_stride(DQK) + acc_stride(DV)) * 4;
    static constexpr size_t LDS_BYTES = NW * RING > MERGE ? NW * RING : MERGE;
    static_assert(LDS_BYTES <= 160 * 1024, "gfx950 LDS");
    static constexpr int WPE = 2 * LDS_BYTES <= 160 * 1024 ? 2 : 1;
    static constexpr int COPIES = WaveCopy<LQ, false>::LOADS + WaveCopy<LO, false>::LOADS + 2;
};
// P enters the dV product as P 2^6: every P above the 1e-6 gate is then in
// fp16's normal range (as in sdpa_f16_dkdv_split.hip).
constexpr float kPScale = 64.f;

template <int DQK, int DV, bool CAUSAL, bool DROP, bool DS, bool P4>
__global__ __launch_bounds__((DkvWaveCfg<DQK, DV>::NT))
__attribute__((amdgpu_waves_per_eu(DkvWaveCfg<DQK, DV>::WPE, DkvWaveCfg<DQK, DV>::WPE)))
void sdpa_bwd_dkdv_f16_wave_kernel(const BwdParams p, const int win) {
    using Cfg = DkvWaveCfg<DQK, DV>;
    constexpr int BKV = Cfg::BKV, BQ = Cfg::BQ, LQ = Cfg::LQ, LO = Cfg::LO, NW = Cfg::NW;
    constexpr int NK = DQK / 16, NV = DV / 16;

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int B = p.s.B, S_q = p.s.S_q, S_kv = p.s.S_kv, D_qk = p.s.D_qk, D_v = p.s.D_v;
    const int tiles = (S_kv + BKV - 1) / BKV;
    int b, kt;
    xcd_map(blockIdx.x, B * tiles, tiles, false, win, b, kt);
    const int k0 = kt * BKV, my_k = k0 + l32;

    const half_t* Kb = static_cast<const half_t*>(p.k) + (size_t)b * S_kv * D_qk;
    const half_t* Vb = static_cast<const half_t*>(p.v) + (size_t)b * S_kv * D_v;
    const RowSrc qsrc = row_src(p.q, (size_t)b * S_q, S_q, D_qk * 2);
    const RowSrc osrc = row_src(p.d_o, (size_t)b * S_q, S_q, D_v * 2);
    const float* stb = (P4 ? p.stats : p.stats2) + (size_t)b * S_q;
    const float* deltab = p.delta + (size_t)b * S_q;

    // query blocks [qb0, nqb); this wave's: qb0 + wave, + NW, ...
    const int qb0 = CAUSAL ? k0 / BQ : 0, nqb = (S_q + BQ - 1) / BQ;
    const uint32_t ringo = (uint32_t)(wave * Cfg::RING), ring = lds_base() + ringo;
    WaveCopy<LQ, false> qc;
    WaveCopy<LO, false> oc;
    qc.init(lane, D_qk * 2, (D_qk + 7) / 8);
    oc.init(lane, D_v * 2, (D_v + 7) / 8);
    auto issue = [&](int qb, uint32_t so) {
        const int q0 = qb * BQ;
        qc.issue(qsrc.shifted(q0), ring + so);
        oc.issue(osrc.shifted(q0), ring + so + (uint32_t)Cfg::QB);
        unsigned char* f = smem + ringo + so + Cfg::QB + Cfg::OB;
        dma4(make_rsrc(stb + q0, (long long)(S_q - q0) * 4), f, lane * 4);
        dma4(make_rsrc(deltab + q0, (long long)(S_q - q0) * 4), f + 256, lane * 4);
    };

    half8 kreg[NK], vreg[NV];
#pragma unroll
    for (int ks = 0; ks < NK; ++ks)
        kreg[ks] = __builtin_bit_cast(half8, load_row_chunk<half_t, !P4>(Kb, my_k, S_kv, 16 * ks + 8 * hh, D_qk, D_qk));
#pragma unroll
    for (int ks = 0; ks < NV; ++ks)
        vreg[ks] = __builtin_bit_cast(half8, load_row_chunk<half_t, !P4>(Vb, my_k, S_kv, 16 * ks + 8 * hh, D_v, D_v));
    prologue_loads_landed();
    if (qb0 + wave < nqb) issue(qb0 + wave, 0);
    // At a 128-wide side, where dS may be stored, as in the split-role kernel:
    // with dropout dS' = dS (1 - p) = P (keep ? dP - delta' : -delta') with
    // delta' = delta (1 - p), and dK is stored with scale / (1 - p).
    // keep_scale 0 (dropout > 1, every element dropped): dP from zero V rows,
    // delta' = delta, so dS' = -P delta.  Else dS itself, which keeps more bits
    // above fp16's smallest normal value: dropout 0.9 with dO ~ 1e-3, error of
    // dK against 64 bits 2.2e-3 with dS', 3.6e-4 with dS.
    constexpr bool SCALED = DQK == 128 || DV == 128;
    static_assert(SCALED || !DS, "stored dS is dS'");
    const float ksc = p.c.keep_scale;
    const bool drop_all = SCALED && DROP && ksc == 0.f;
    if (drop_all) {
#pragma unroll
        for (int ks = 0; ks < NV; ++ks) vreg[ks] = half8{};
    }
    const float rksc = SCALED && DROP && !drop_all ? 1.f / ksc : 1.f;
    const float sl2 = p.c.scale_log2;
    const uint64_t row_step = (uint64_t)S_kv * kLcgMul;
    uint64_t st = DROP ? lcg_state(p.c.seed_offset, (uint64_t)b * S_q + (uint64_t)((qb0 + wave) * BQ + 4 * hh),
                                   (uint64_t)S_kv, my_k)
                       : 0;
    const uint32_t thr = p.c.drop_threshold;
    SwzLane<LQ> swQ;
    SwzLane<LO> swO;
    swQ.init(lane);
    swO.init(lane);
    floatx16 dkacc[DQK / 32], dvacc[DV / 32];
#pragma unroll
    for (int dt = 0; dt < DQK / 32; ++dt) dkacc[dt] = floatx16{};
#pragma unroll
    for (int dt = 0; dt < DV / 32; ++dt) dvacc[dt] = floatx16{};
    const DsLayout dsl(S_q, S_kv, CAUSAL);

    uint32_t so = 0;
    for (int qb = qb0 + wave; qb < nqb; qb += NW, so ^= (uint32_t)Cfg::STAGE) {
        lds_reads_done();
        if (qb + NW < nqb) {
            issue(qb + NW, so ^ (uint32_t)Cfg::STAGE);
            wait_copies<Cfg::COPIES>();
        } else {
            wait_copies<0>();
        }
        const int q0 = qb * BQ;
        const uint32_t qbase = ringo + so, obase = qbase + (uint32_t)Cfg::QB;
        const float* Fs = reinterpret_cast<const float*>(smem + obase + Cfg::OB);
        floatx16 s = floatx16{}, dp = floatx16{};
#pragma unroll
        for (int ks = 0; ks < NK; ++ks) s = mfma_f16(keep4<P4>(lds_row<LQ>(qbase + swQ.row, ks, 0), ks, hh, D_qk), kreg[ks], s);
#pragma unroll
        for (int ks = 0; ks < NV; ++ks) dp = mfma_f16(keep4<P4>(lds_row<LO>(obase + swO.row, ks, 0), ks, hh, D_v), vreg[ks], dp);
        // rows past S_q (their zero stats2 would make P = 2^kGateShift) and,
        // causal, keys after the query
        const bool mask = q0 + BQ > S_q || (CAUSAL && q0 < k0 + BKV - 1);
        uint32_t wp[8], wd[8];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const floatx4 st4 = *reinterpret_cast<const floatx4*>(Fs + 8 * g + 4 * hh);
            const floatx4 de4 = *reinterpret_cast<const floatx4*>(Fs + 64 + 8 * g + 4 * hh);
            float pk4[4], ds4[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int r = 4 * g + e;
                float x = __builtin_fmaf(s[r], sl2, P4 ? -(st4[e] * kLog2e) : -st4[e]);
                if (mask) {
                    const int q = q0 + 8 * g + 4 * hh + e;
                    if (q >= S_q || (CAUSAL && my_k > q)) x = -INFINITY;
                }
                const float pr = gated<P4>(x);
                float pk = pr * kPScale, t;
                if constexpr (DROP) {
                    const float de = SCALED ? de4[e] * rksc : de4[e];
                    const bool keep = lcg_keep(st + (uint64_t)(8 * g + e) * row_step, thr);
                    pk = keep ? pk : 0.f;
                    t = keep ? (SCALED ? dp[r] - de : __builtin_fmaf(dp[r], ksc, -de)) : -de;
                } else {
                    t = dp[r] - de4[e];
                }
                pk4[e] = pk;
                ds4[e] = pr * t;
            }
            wp[2 * g] = pack_h2(pk4[0], pk4[1]);
            wp[2 * g + 1] = pack_h2(pk4[2], pk4[3]);
            wd[2 * g] = pack_h2(ds4[0], ds4[1]);
            wd[2 * g + 1] = pack_h2(ds4[2], ds4[3]);
        }
        if constexpr (DROP) st += (uint64_t)(NW * BQ) * row_step;
        const half8 p0 = half8_of(wp[0], wp[1], wp[2], wp[3]), p1 = half8_of(wp[4], wp[5], wp[6], wp[7]);
        half8 d0 = half8_of(wd[0], wd[1], wd[2], wd[3]), d1 = half8_of(wd[4], wd[5], wd[6], wd[7]);
#pragma unroll
        for (int dt = 0; dt < DV / 32; ++dt) {
            dvacc[dt] = mfma_f16(lds_tr<LO>(obase + swO.tr0, obase + swO.tr1, dt, 0), p0, dvacc[dt]);
            dvacc[dt] = mfma_f16(lds_tr<LO>(obase + swO.tr0, obase + swO.tr1, dt, 16), p1, dvacc[dt]);
        }
#pragma unroll
        for (int dt = 0; dt < DQK / 32; ++dt) {
            dkacc[dt] = mfma_f16(lds_tr<LQ>(qbase + swQ.tr0, qbase + swQ.tr1, dt, 0), d0, dkacc[dt]);
            dkacc[dt] = mfma_f16(lds_tr<LQ>(qbase + swQ.tr0, qbase + swQ.tr1, dt, 16), d1, dkacc[dt]);
        }
        if constexpr (DS) {
            // sub-tile q0 of key group k0 / 32 of chunk (k0 / 128, q0 / 64);
            // zero for keys past S_kv (dQ reads them unmasked)
            if (my_k >= S_kv) {
                d0 = half8{};
                d1 = half8{};
            }
            unsigned char* dst = static_cast<unsigned char*>(p.ds) + dsl.offset(b, k0 / DsLayout::KT, q0 / DsLayout::QBK) +
                                 (q0 / 32 % 2) * 8192 + (k0 / 32 % 4) * 2048;
            *reinterpret_cast<half8*>(dst + DsLayout::slot(l32, hh)) = d0;
            *reinterpret_cast<half8*>(dst + DsLayout::slot(l32, 2 + hh)) = d1;
        }
    }

    __syncthreads();  // every ring has been read
    float* mk = reinterpret_cast<float*>(smem);
    float* mv = mk + NW * BKV * acc_stride(DQK);
    acc_to_lds<DQK>(mk, wave * BKV + l32, dkacc, hh);
    acc_to_lds<DV>(mv, wave * BKV + l32, dvacc, hh);
    __syncthreads();
    const size_t krow0 = (size_t)b * S_kv + k0;
    const float fk = SCALED && DROP && !drop_all ? p.c.scale * ksc : p.c.scale, fv = ksc * (1.f / kPScale);
    sum_waves<NW, BKV, DQK>(mk, tid, S_kv - k0, D_qk, [&](int row, int c, const floatx4& sum) {
        *reinterpret_cast<half4*>(static_cast<half_t*>(p.dk) + (krow0 + row) * D_qk + c) = scaled_h4(sum, fk);
    });
    sum_waves<NW, BKV, DV>(mv, tid, S_kv - k0, D_v, [&](int row, int c, const floatx4& sum) {
        *reinterpret_cast<half4*>(static_cast<half_t*>(p.dv) + (krow0 + row) * D_v + c) = scaled_h4(sum, fv);
    });
}

// ---------------------------------------------------------------------------
// dQ of one stored query block (64 queries) from the stored dS'
// ---------------------------------------------------------------------------
template <int DQK>
struct DqDsWaveCfg {
    static constexpr int NW = kSmallWaves, NT = 64 * NW, BM = DsLayout::QBK, BN = 32;
    static constexpr int LK = DQK / 8;
    static constexpr int KB = BN * DQK * 2, SB = BN * 64;  // K tile; one 32-query dS' tile
    static constexpr int STAGE = KB + 2 * SB, RING = 2 * STAGE;
    static constexpr int MERGE = NW * BM * acc_stride(DQK) * 4;
    static constexpr size_t LDS_BYTES = NW * RING > MERGE ? NW * RING : MERGE;
    static_assert(LDS_BYTES <= 160 * 1024, "gfx950 LDS");
    static constexpr int WPE = 2 * LDS_BYTES <= 160 * 1024 ? 2 : 1;
    static constexpr int COPIES = WaveCopy<LK, true>::LOADS + 4;
};

template <int DQK, bool CAUSAL>
__global__ __launch_bounds__((DqDsWaveCfg<DQK>::NT))
__attribute__((amdgpu_waves_per_eu(DqDsWaveCfg<DQK>::WPE, DqDsWaveCfg<DQK>::WPE)))
void sdpa_bwd_dq_ds_f16_wave_kernel(const BwdParams p, const int win) {
    using Cfg = DqDsWaveCfg<DQK>;
    constexpr int BM = Cfg::BM, BN = Cfg::BN, LK = Cfg::LK, NW = Cfg::NW, NDT = DQK / 32;

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int B = p.s.B, S_q = p.s.S_q, S_kv = p.s.S_kv, D_qk = p.s.D_qk;
    const int tiles = (S_q + BM - 1) / BM;
    int b, qb;
    xcd_map(blockIdx.x, B * tiles, tiles, CAUSAL, win, b, qb);
    const int q0 = qb * BM;
    const int pq = 8 * ((l32 >> 2) & 3) + 4 * (l32 >> 4) + (l32 & 3);  // stored position -> query
    const DsLayout dsl(S_q, S_kv, CAUSAL);
    const unsigned char* dsb = static_cast<const unsigned char*>(p.ds);
    const RowSrc ksrc = row_src(p.k, (size_t)b * S_kv, S_kv, D_qk * 2);
    const uint32_t ringo = (uint32_t)(wave * Cfg::RING), ring = lds_base() + ringo;
    WaveCopy<LK, true> kc;
    kc.init(lane, D_qk * 2, (D_qk + 7) / 8);
    const int nblk = (min(S_kv, CAUSAL ? q0 + BM : S_kv) + BN - 1) / BN;
    // A sub-tile the dK/dV kernel did not store (its queries all before the
    // key group, or past S_q) is copied from an empty range: zeros.
    auto issue = [&](int blk, uint32_t so) {
        const int kv0 = blk * BN;
        kc.issue(ksrc.shifted(kv0), ring + so);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int qs = q0 + 32 * t;
            const bool stored = qs < S_q && !(CAUSAL && qs + 31 < kv0);
            const unsigned char* src = dsb + (stored ? dsl.offset(b, kv0 / DsLayout::KT, qb) : 0) + t * 8192 +
                                       (kv0 % DsLayout::KT) * 64;
            const rsrc_t rs = make_rsrc(uniform_ptr(src), stored ? Cfg::SB : 0);
            const uint32_t m0 = ring + so + (uint32_t)(Cfg::KB + Cfg::SB * t);
            dma16_at(rs, m0, (uint32_t)lane * 16);
            dma16_at(rs, m0 + 1024, 1024u + (uint32_t)lane * 16);
        }
    };
    if (wave < nblk) issue(wave, 0);

    floatx16 acc[2][NDT];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) acc[t][dt] = floatx16{};
    const uint32_t kl = ring + tr_lane_off<LK>(lane);  // K^T
    uint32_t sl0, sl8;  // dS'^T: the transposed read at its place in the stored tile (sdpa_f16_dq_ds.hip)
    {
        const int g16 = lane >> 4, i16 = lane & 15;
        const int tr_row = 4 * (g16 >> 1) + (i16 >> 2), c = 2 * (g16 & 1) + ((i16 & 3) >> 1), sub = 8 * (i16 & 1);
        const int pl = 2 * (c & 1) + (c >> 1);
        const uint32_t base = ring + (uint32_t)(Cfg::KB + sub);
        sl0 = base + (uint32_t)DsLayout::slot(tr_row, pl);
        sl8 = base + (uint32_t)DsLayout::slot(tr_row + 8, pl);
    }
    uint32_t so = 0;
    for (int blk = wave; blk < nblk; blk += NW, so ^= (uint32_t)Cfg::STAGE) {
        lds_reads_done();
        if (blk + NW < nblk) {
            issue(blk + NW, so ^ (uint32_t)Cfg::STAGE);
            wait_copies<Cfg::COPIES>();
        } else {
            wait_copies<0>();
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            half8 bs[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const uint32_t a = so + (uint32_t)(Cfg::SB * t + 256 * j);
                bs[t] = ld_tr8(sl0 + a, sl8 + a);
            }
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) {
                const uint32_t a = (kl ^ (uint32_t)(64 * dt)) + so;
                const half8 ak = ld_tr8(a + 256u * LK * j, a + 16u * LK * (16 * j + 8));
#pragma unroll
                for (int t = 0; t < 2; ++t) acc[t][dt] = mfma_f16(ak, bs[t], acc[t][dt]);
            }
        }
    }

    __syncthreads();  // every ring has been read
    float* m = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int t = 0; t < 2; ++t) acc_to_lds<DQK>(m, wave * BM + 32 * t + pq, acc[t], hh);
    __syncthreads();
    // dS' = dS (1-p) with dropout; every element dropped (keep_scale 0): dS' = dS
    const float f = (p.c.use_dropout && p.c.keep_scale != 0.f) ? p.c.scale * p.c.keep_scale : p.c.scale;
    const size_t grow0 = (size_t)b * S_q + q0;
    sum_waves<NW, BM, DQK>(m, tid, S_q - q0, D_qk, [&](int row, int c, const floatx4& sum) {
        *reinterpret_cast<half4*>(static_cast<half_t*>(p.dq) + (grow0 + row) * D_qk + c) = scaled_h4(sum, f);
    });
}

}  // namespace

hipError_t launch_bwd_dq_f16_wave(const BwdParams& p, hipStream_t stream) {
    const int B = p.s.B, S_q = p.s.S_q;
    if (B == 0 || S_q == 0) return hipSuccess;
    return with_dim(p.s.D_qk, [&](auto dqk) {
        return with_dim(p.s.D_v, [&](auto dv) {
            return with_bool(p.c.causal != 0, [&](auto c) {
                return with_bool(p.c.use_dropout != 0, [&](auto d) {
                    constexpr int DQK = decltype(dqk)::value, DV = decltype(dv)::value;
                    if constexpr (DQK <= 64 && DV <= 64) {
                        using Cfg = DqWaveCfg<DQK, DV>;
                        const long long n = (long long)((S_q + Cfg::BM - 1) / Cfg::BM) * p.parts * B;
                        constexpr bool CA = decltype(c)::value, DR = decltype(d)::value;
                        const int win = row_window((size_t)p.s.S_kv * (DQK + DV) * 2);
                        hipError_t err;
                        if (p.s.D_qk % 8 == 0 && p.s.D_v % 8 == 0)
                            err = launch_kernel<sdpa_bwd_dq_f16_wave_kernel<DQK, DV, CA, DR, false>>(
                                (unsigned)n, Cfg::NT, Cfg::LDS_BYTES, stream, p, win);
                        else
                            err = launch_kernel<sdpa_bwd_dq_f16_wave_kernel<DQK, DV, CA, DR, true>>(
                                (unsigned)n, Cfg::NT, Cfg::LDS_BYTES, stream, p, win);
                        if (err == hipSuccess && p.parts > 1) {
                            const long long th = (long long)B * S_q * (p.s.D_qk / 4);
                            err = launch_kernel<sdpa_bwd_dq_merge_f16_kernel>((unsigned)((th + 255) / 256), 256, 0, stream, p);
                        }
                        return err;
                    } else {
                        return hipErrorInvalidValue;
                    }
                });
            });
        });
    });
}

hipError_t launch_bwd_dkdv_f16_wave(const BwdParams& p, hipStream_t stream) {
    const int B = p.s.B, S_kv = p.s.S_kv;
    if (B == 0 || S_kv == 0) return hipSuccess;
    return with_dim(p.s.D_qk, [&](auto dqk) {
        return with_dim(p.s.D_v, [&](auto dv) {
            return with_bool(p.c.causal != 0, [&](auto c) {
                return with_bool(p.c.use_dropout != 0, [&](auto d) {
                    constexpr int DQK = decltype(dqk)::value, DV = decltype(dv)::value;
                    constexpr bool CA = decltype(c)::value, DR = decltype(d)::value;
                    using Cfg = DkvWaveCfg<DQK, DV>;
                    const unsigned n = (unsigned)((long long)((S_kv + Cfg::BKV - 1) / Cfg::BKV) * B);
                    const int win = row_window((size_t)p.s.S_q * (DQK + DV) * 2);
                    if constexpr (DQK == 128 || DV == 128) {
                        if (p.ds)
                            return launch_kernel<sdpa_bwd_dkdv_f16_wave_kernel<DQK, DV, CA, DR, true, false>>(
                                n, Cfg::NT, Cfg::LDS_BYTES, stream, p, win);
                    }
                    if constexpr (DQK <= 64 && DV <= 64) {
                        if (p.s.D_qk % 8 != 0 || p.s.D_v % 8 != 0)
                            return launch_kernel<sdpa_bwd_dkdv_f16_wave_kernel<DQK, DV, CA, DR, false, true>>(
                                n, Cfg::NT, Cfg::LDS_BYTES, stream, p, win);
                    }
                    return launch_kernel<sdpa_bwd_dkdv_f16_wave_kernel<DQK, DV, CA, DR, false, false>>(
                        n, Cfg::NT, Cfg::LDS_BYTES, stream, p, win);
                });
            });
        });
    });
}

hipError_t launch_bwd_dq_ds_f16_wave(const BwdParams& p, hipStream_t stream) {
    const int B = p.s.B, S_q = p.s.S_q;
    if (B == 0 || S_q == 0) return hipSuccess;
    if (!p.ds) return hipErrorInvalidValue;
    return with_dim(p.s.D_qk, [&](auto dqk) {
        return with_bool(p.c.causal != 0, [&](auto c) {
            using Cfg = DqDsWaveCfg<decltype(dqk)::value>;
            const long long n = (long long)((S_q + Cfg::BM - 1) / Cfg::BM) * B;
            return launch_kernel<sdpa_bwd_dq_ds_f16_wave_kernel<decltype(dqk)::value, decltype(c)::value>>(
                (unsigned)n, Cfg::NT, Cfg::LDS_BYTES, stream, p, row_window((size_t)p.s.S_kv * decltype(dqk)::value * 2));
        });
    });
}

}  // namespace sdpa
