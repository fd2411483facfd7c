// sdpa_f32_dq_ds.hip -- the dS path of the fp32 SdpaGrad for gfx950: dQ as a
// product with the dS the fp32 dK/dV kernel stored (DsLayout32), instead
// of the dQ kernel that forms S, P, dP and dS once more (sdpa_bwd.hip).
//
// Order of the path (sdpa_capi.hip):
//   1. row kernel  -- delta (and stats2) per query row into the workspace, as
//                     the other path's dQ kernel writes them first;
//   2. dK/dV       -- sdpa_f32_dkdv.hip with p.ds set: its dS
//                     role stores every dS it forms;
//   3. dQ          -- dQ^T = K^T dS^T per 32 queries, scaled once at the store.
//
// Element semantics (sdpa/sdpa_bwd.cu.cc:291-327): dQ_i = scale sum_j dS_ij
// K_j with dS as the dK/dV kernel forms it (P gated at 1e-6, the dropout
// decision, dP scaled by 1/(1-p) for kept elements).
#include <type_traits>

#include "sdpa_bf3.h"
#include "sdpa_launch.h"
#include "sdpa_params.h"

namespace sdpa {
namespace {

// ---------------------------------------------------------------------------
// Row values.  Lane = query row, hh = half of the features: delta = sum_d dO
// O summed as the fp32 dQ kernel's prologue sums it (its lane, feature and
// fma order), so that both paths hand the dK/dV kernel the same delta and dK,
// dV are bit-identical between them.  stats2 as that prologue writes it.
// ---------------------------------------------------------------------------
template <int DV>
__global__ __launch_bounds__(256) void sdpa_bwd_rows_f32_kernel(const BwdParams p) {
    constexpr int HV = DV / 2;
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5, wave = tid >> 6;
    const int S_q = p.s.S_q, D_v = p.s.D_v;
    const int tiles = (S_q + 127) / 128;
    const int b = (int)(blockIdx.x / (unsigned)tiles), qt = (int)(blockIdx.x % (unsigned)tiles);
    const int my_q = qt * 128 + 32 * wave + l32;
    const size_t row_q = (size_t)b * S_q + my_q;
    const float* Ob = static_cast<const float*>(p.o) + (size_t)b * S_q * D_v;
    const float* dOb = static_cast<const float*>(p.d_o) + (size_t)b * S_q * D_v;
    float dpart = 0.f;
#pragma unroll
    for (int u = 0; u < HV / 4; ++u) {
        const floatx4 f = __builtin_bit_cast(floatx4, load_row_chunk<float, true>(dOb, my_q, S_q, HV * hh + 4 * u, D_v, D_v));
        const floatx4 o = __builtin_bit_cast(floatx4, load_row_chunk<float, true>(Ob, my_q, S_q, HV * hh + 4 * u, D_v, D_v));
#pragma unroll
        for (int e = 0; e < 4; ++e) dpart += f[e] * o[e];
    }
    const float delta = xhalf_sum(dpart);
    if (my_q < S_q && hh == 0) {
        const float stats2 = p.stats[row_q] * kLog2e;
        p.delta[row_q] = delta;
        p.stats2[row_q] = stats2 + kGateShift;
    }
}

// ---------------------------------------------------------------------------
// dQ from the stored dS, on the bf16 matrix cores (sdpa_bf3.h).  128 queries
// per workgroup, a stored query block of 32 for each group of waves; the two
// waves of a group, on one SIMD, share its keys (one stored key group of 32
// per 64-key step each; their sums are added through LDS at the end).  The K
// tile is staged through registers and cut into its parts on the way; each
// wave's 4 KB dS tile is copied as it lies, read per key as stored (lane =
// query position) and cut in registers.  Lane l32 stores query pi(l32).
//
// B 64, S_q 512, S_kv 16384, D_qk 128 (2.1 GB of dS): 1.08 ms on
// v_mfma_f32_32x32x2_f32 (81% busy), 0.79 ms here; error of dQ against
// 64 bits 2.5e-6 -> 1.8e-6.
// ---------------------------------------------------------------------------
template <int DQK>
struct DqDs32Cfg {
    static constexpr int NT = 512, BM = 128, BN = 64;
    using KT = Bf3Tile<BN, DQK / 8>;
    static constexpr int SB = 4096;  // one wave's dS tile
    static constexpr int SOFF = 2 * KT::BYTES;
    static constexpr int OS = DQK + 4, MERGE = BM * OS * 4;  // after the loop
    static constexpr size_t LDS_BYTES = SOFF + 16 * SB > MERGE ? SOFF + 16 * SB : MERGE;
    static_assert(LDS_BYTES <= 160 * 1024, "gfx950 LDS");
};

template <int DQK, bool CAUSAL>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void sdpa_bwd_dq_ds_f32_kernel(const BwdParams p, const int win) {
    using Cfg = DqDs32Cfg<DQK>;
    using KT = typename Cfg::KT;
    constexpr int BM = Cfg::BM, BN = Cfg::BN, LK = DQK / 8, NDT = DQK / 32;
    static_assert(DsLayout32::KT % BN == 0 && DsLayout32::QBK == 32, "steps tile the stored key groups");

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wq = wave & 3, wk = wave >> 2;
    const int B = p.s.B, S_q = p.s.S_q, S_kv = p.s.S_kv, D_qk = p.s.D_qk;
    const int tiles = (S_q + BM - 1) / BM;
    int b, qt;
    const int id = tile_id();
    if (id >= B * tiles) return;
    xcd_map(id, B * tiles, tiles, CAUSAL, win, b, qt);
    const int qw0 = qt * BM + 32 * wq, qb = qw0 / DsLayout32::QBK;
    const int pq = 8 * ((l32 >> 2) & 3) + 4 * (l32 >> 4) + (l32 & 3);  // stored position -> query
    const DsLayout32 dsl(S_q, S_kv, CAUSAL);
    const unsigned char* dsb = static_cast<const unsigned char*>(p.ds);
    const float* Kb = static_cast<const float*>(p.k) + (size_t)b * S_kv * D_qk;
    const int nsteps = ((CAUSAL ? min(S_kv, qt * BM + BM) : S_kv) + BN - 1) / BN;

    // The dK/dV kernel stored this wave's block at the key group kv0 under
    // the same predicate (its `live`).
    auto live = [&](int kv0) { return qw0 < S_q && kv0 < S_kv && !(CAUSAL && qw0 + 31 < kv0); };
    const uint32_t s0 = (uint32_t)(Cfg::SOFF + 2 * Cfg::SB * wave);  // this wave's two dS stages
    auto copy_ds = [&](int step) {
        const int kv0 = step * BN + 32 * wk;
        if (!live(kv0)) return;
        const unsigned char* src = dsb + dsl.offset(b, kv0 / DsLayout32::KT, qb) + ((kv0 % DsLayout32::KT) / 32) * 4096;
        const rsrc_t rs = make_rsrc(uniform_ptr(src), Cfg::SB);
        const uint32_t m0 = lds_base() + s0 + (uint32_t)((step & 1) * Cfg::SB);
        // dS is read once: non-temporal
#pragma unroll
        for (int u = 0; u < 4; ++u) dma16_at_nt(rs, m0 + 1024u * u, (uint32_t)(16 * lane + 1024 * u));
    };
    Bf3Stage<BN, DQK, Cfg::NT, true> kst;
    auto load_k = [&](int step) { kst.load(Kb, step * BN, S_kv - step * BN, D_qk, D_qk, tid); };
    auto store_k = [&](int step) { kst.store(smem + (step & 1) * KT::BYTES, tid); };

    SwzLane<LK> swK;
    swK.init(lane);
    // dS of key r, position l32 sits at slot32(r, l32) = base + 16 (r ^ (u + 4
    // h)); for the keys 8 i + 4 hh + e of an operand the XOR term stays below
    // 8: one lane base per e, 128 i as an immediate
    int sbase[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) sbase[e] = DsLayout32::slot32(4 * hh + e, l32);
    floatx16 acc[NDT];

    // INF: again, for infinities in dS (sdpa_bf3.h)
    auto pass = [&](auto inf) {
        constexpr bool INF = decltype(inf)::value;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) acc[dt] = floatx16{};
        if (nsteps > 0) {
            copy_ds(0);
            load_k(0);
            store_k(0);
            wait_vm();
            if (nsteps > 1) load_k(1);
        }
        __syncthreads();
        for (int step = 0; step < nsteps; ++step) {
            // the other stages were released at the last barrier
            if (step + 1 < nsteps) copy_ds(step + 1);
            if (live(step * BN + 32 * wk)) {
                const uint32_t ks0 = (uint32_t)((step & 1) * KT::BYTES);
                const unsigned char* Ss = smem + s0 + (step & 1) * Cfg::SB;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const Bf3 ds = cut8<INF>([&](int i) {
                        return *reinterpret_cast<const float*>(Ss + sbase[i & 3] + 128 * (2 * j + (i >> 2)));
                    });
#pragma unroll
                    for (int dt = 0; dt < NDT; ++dt)
                        acc[dt] = mfma_bf3<INF>(KT::tr(ks0 + swK.tr0, ks0 + swK.tr1, dt, 32 * wk + 16 * j), ds, acc[dt]);
                }
            }
            if (step + 1 < nsteps) store_k(step + 1);
            wait_vm();  // the next step's dS
            if (step + 2 < nsteps) load_k(step + 2);
            __syncthreads();
        }
    };
    pass(std::false_type{});
    if (workgroup_any_nan<Cfg::NT / 64>(acc, tid)) pass(std::true_type{});

    float* m = reinterpret_cast<float*>(smem) + (32 * wq + l32) * Cfg::OS;
    if (wk == 1) store_rows_f32<DQK, true>(m, acc, 1.f, hh, DQK);
    __syncthreads();
    const int my_q = qw0 + pq;
    if (wk == 1 || my_q >= S_q) return;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const floatx4 x = *reinterpret_cast<const floatx4*>(m + 32 * dt + 8 * g + 4 * hh);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[dt][4 * g + e] += x[e];
        }
    store_rows_f32<DQK, true>(static_cast<float*>(p.dq) + ((size_t)b * S_q + my_q) * D_qk, acc, p.c.scale, hh, D_qk);
}

}  // namespace

hipError_t launch_bwd_rows_f32(const BwdParams& p, hipStream_t stream) {
    const int B = p.s.B, S_q = p.s.S_q;
    if (B == 0 || S_q == 0) return hipSuccess;
    const long long n = (long long)((S_q + 127) / 128) * B;
    if (n > 0x7FFFFFFFLL) return hipErrorInvalidValue;
    return with_dim(p.s.D_v, [&](auto dv) {
        constexpr int DV = decltype(dv)::value;
        return launch_kernel<sdpa_bwd_rows_f32_kernel<DV>>((unsigned)n, 256, 0, stream, p);
    });
}

hipError_t launch_bwd_dq_ds_f32(const BwdParams& p, hipStream_t stream) {
    const int B = p.s.B, S_q = p.s.S_q;
    if (B == 0 || S_q == 0) return hipSuccess;
    if (!p.ds) return hipErrorInvalidValue;
    return with_dim(p.s.D_qk, [&](auto dqk) {
        return with_bool(p.c.causal != 0, [&](auto c) {
            constexpr int DQK = decltype(dqk)::value;
            using Cfg = DqDs32Cfg<DQK>;
            const long long n = (long long)((S_q + Cfg::BM - 1) / Cfg::BM) * B;
            return launch_kernel<sdpa_bwd_dq_ds_f32_kernel<DQK, decltype(c)::value>>(
                tile_grid(n, Cfg::NT), Cfg::NT, Cfg::LDS_BYTES, stream, p, row_window((size_t)p.s.S_kv * DQK * 4));
        });
    });
}

}  // namespace sdpa
