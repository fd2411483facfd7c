// sdpa_f32_dkdv.hip -- fp32 SdpaGrad dK/dV kernel for gfx950, its products on
// the bf16 matrix cores (sdpa_bf3.h).
//
// Replaces FlashAttnBwdKernel_KV for float (sdpa/sdpa_bwd.cu.cc:13-213);
// element semantics as in sdpa_bwd.hip.  Eight waves over 128 keys: each
// group of 32 keys has two, on one SIMD, as in sdpa_f16_dkdv_split.hip:
//   P role:  S = Q K^T, P~, dV^T += dO^T P~   (K's parts in registers)
//   dS role: dP = dO V^T, dS, dK^T += Q^T dS  (V's parts in registers)
// Q/dO blocks of 32 queries are staged through registers into two LDS stages,
// cut into their bf16 parts on the way.  Both roles work on the same block:
// in its first half S and P beside dP and the dS role's share of the staging,
// then (P, with the dropout decision in its sign, has gone through LDS) dV and
// the P role's share beside dS and dK.  The query blocks of a tile may be
// divided over workgroups (bwd_parts), whose sums a second kernel adds.
//
// What bounds it: VALU work (cutting, elements) that overlaps the MFMAs in
// part; the matrix cores are busy 46%.  B 64, S_q 512, D 128/64, with the dS
// stores: 1.19 ms at 8192 keys, 1.87 ms on v_mfma_f32_32x32x2_f32 at 8224 (70%
// busy; sdpa_f32_chain.hip, which takes over there), error of dK against 64
// bits 8.2e-7 and 9.1e-7; D 64 without them 0.82 and 1.33 ms.  The dS role one
// block behind (three stages, one barrier a block) was 4% slower.
#include <type_traits>

#include "sdpa_bf3.h"
#include "sdpa_launch.h"
#include "sdpa_params.h"
#include "sdpa_parts.h"

namespace sdpa {
namespace {

template <int DQK, int DV>
struct DkvBf3Cfg {
    static constexpr int NT = 512, BKV = 128, BQ = 32;
    using QT = Bf3Tile<BQ, DQK / 8>;
    using OT = Bf3Tile<BQ, DV / 8>;
    static constexpr int FB = 2 * BQ * 4;                    // stats log2(e) and delta of the block's rows
    static constexpr int STAGE = QT::BYTES + OT::BYTES + FB;
    static constexpr int XB = 4 * 32 * 32 * 4;               // P of 4 key groups x 32 queries
    static constexpr size_t LDS_BYTES = 2 * STAGE + XB;
    static_assert(LDS_BYTES <= 160 * 1024, "gfx950 LDS");
};

template <int DQK, int DV, bool VEC, bool DROP, bool DS>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void sdpa_bwd_dkdv_f32_bf3_kernel(const BwdParams p, const int win) {
    using Cfg = DkvBf3Cfg<DQK, DV>;
    using QT = typename Cfg::QT;
    using OT = typename Cfg::OT;
    constexpr int BKV = Cfg::BKV, BQ = Cfg::BQ, LQ = DQK / 8, LO = DV / 8;

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kw = wave & 3;
    const int B = p.s.B, S_q = p.s.S_q, S_kv = p.s.S_kv, D_qk = p.s.D_qk, D_v = p.s.D_v;
    const bool causal = p.c.causal != 0;
    const int np = p.kv_parts, items = (S_kv + BKV - 1) / BKV * np;
    int b, it;
    const int id = tile_id();
    if (id >= B * items) return;
    xcd_map(id, B * items, items, false, win, b, it);
    const int kt = it / np, part = it - kt * np;
    const int k0 = kt * BKV, kw0 = k0 + kw * 32, my_k = kw0 + l32;
    const bool key_ok = my_k < S_kv, wave_live = kw0 < S_kv;

    const float* Qb = static_cast<const float*>(p.q) + (size_t)b * S_q * D_qk;
    const float* dOb = static_cast<const float*>(p.d_o) + (size_t)b * S_q * D_v;
    const float* statsb = p.stats + (size_t)b * S_q;
    const float* deltab = p.delta + (size_t)b * S_q;
    // this part's query blocks [qb0, nqb) of those that see the tile
    const int qfirst = causal ? min(k0, S_q) / BQ : 0, qblocks = (S_q + BQ - 1) / BQ - qfirst;
    const int qb0 = qfirst + part_begin(qblocks, part, np), nqb = qfirst + part_begin(qblocks, part + 1, np);
    // a block is skipped by both roles when the key group sees none of it
    auto live = [&](int q0) { return wave_live && (!causal || q0 + BQ - 1 >= kw0); };

    // The registers hold the next block between load and store.
    Bf3Stage<BQ, DQK, Cfg::NT, VEC> qst;
    Bf3Stage<BQ, DV, Cfg::NT, VEC> ost;
    float fpre = 0.f;
    auto load_block = [&](int qb) {
        const int q0 = qb * BQ;
        qst.load(Qb, q0, S_q - q0, D_qk, D_qk, tid);
        ost.load(dOb, q0, S_q - q0, D_v, D_v, tid);
        if (tid < 2 * BQ) {
            const int r = q0 + (tid & (BQ - 1));
            if (tid < BQ) fpre = r < S_q ? statsb[r] * kLog2e : INFINITY;
            else fpre = r < S_q ? deltab[r] : 0.f;
        }
    };
    auto store_block = [&](int qb, auto inf) {
        constexpr bool INF = decltype(inf)::value;
        unsigned char* st = smem + ((qb - qb0) & 1) * Cfg::STAGE;
        qst.store(st, tid);
        ost.template store<INF>(st + QT::BYTES, tid);
        if (tid < 2 * BQ) reinterpret_cast<float*>(st + QT::BYTES + OT::BYTES)[tid] = fpre;
    };
    auto stage_next = [&](int qb, auto inf) {
        if (qb + 1 < nqb) {
            store_block(qb + 1, inf);
            if (qb + 2 < nqb) load_block(qb + 2);
        }
    };
    float* xs = reinterpret_cast<float*>(smem + 2 * Cfg::STAGE) + kw * 1024;  // this key group's P
    auto stage_first = [&](auto inf) {
        if (qb0 < nqb) {
            load_block(qb0);
            store_block(qb0, inf);
            if (qb0 + 1 < nqb) load_block(qb0 + 1);
        }
    };
    // Each role passes over the blocks; INF: again, for infinities in dO, V or
    // dS (sdpa_bf3.h), which either role may find
    stage_first(std::false_type{});
    SwzLane<LQ> swQ;
    SwzLane<LO> swO;
    swQ.init(lane);
    swO.init(lane);

    if (wave < 4) {
        // ------------------------------------------------------------ P role
        Bf3 k[DQK / 16];
        load_row_bf3<DQK, VEC>(k, static_cast<const float*>(p.k) + (size_t)b * S_kv * D_qk, my_k, S_kv, D_qk, hh);
        const float sl2 = p.c.scale_log2;
        const uint64_t st_base = DROP ? lcg_state(p.c.seed_offset, (uint64_t)b * S_q + 4 * hh, (uint64_t)S_kv, my_k) : 0;
        const uint64_t row_step = (uint64_t)S_kv * kLcgMul;
        const uint32_t thr = p.c.drop_threshold;
        floatx16 dv[DV / 32];
        auto pass = [&](auto inf) {
            constexpr bool INF = decltype(inf)::value;
            if constexpr (INF) stage_first(inf);
#pragma unroll
            for (int dt = 0; dt < DV / 32; ++dt) dv[dt] = floatx16{};
            __syncthreads();
            for (int qb = qb0; qb < nqb; ++qb) {
                const int q0 = qb * BQ;
                const uint32_t qs = (uint32_t)(((qb - qb0) & 1) * Cfg::STAGE), os = qs + (uint32_t)QT::BYTES;
                const bool on = live(q0);
                floatx16 s = floatx16{};
                if (on) {
#pragma unroll
                    for (int ks = 0; ks < DQK / 16; ++ks) s = mfma_bf3(QT::row(qs + swQ.row, ks, 0), k[ks], s);
                    const float* Fs = reinterpret_cast<const float*>(smem + os + OT::BYTES);
                    if (kw0 + 31 >= S_kv || (causal && q0 < kw0 + 31)) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const int q = q0 + 8 * (r >> 2) + 4 * hh + (r & 3);
                            if (!key_ok || (causal && my_k > q)) s[r] = sl2 < 0.f ? INFINITY : -INFINITY;
                        }
                    }
                    float sum = 0.f;
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const floatx4 st4 = *reinterpret_cast<const floatx4*>(Fs + 8 * g + 4 * hh);
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            s[4 * g + e] = fast_exp2(__builtin_fmaf(s[4 * g + e], sl2, -st4[e]));
                            sum += s[4 * g + e];
                        }
                    }
                    if (wave_any(sum != sum)) {  // scores of -inf (see sdpa_f32_fwd.hip)
                        lds_read_again();
                        floatx16 h = floatx16{};
#pragma unroll
                        for (int ks = 0; ks < DQK / 16; ++ks) h = mfma_bf16(QT::row(qs + swQ.row, ks, 0).p[0], k[ks].p[0], h);
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                            if (h[r] * sl2 == -INFINITY) s[r] = 0.f;
                    }
                    const uint64_t st_blk = DROP ? st_base + (uint64_t)q0 * row_step : 0;
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        floatx4 xv;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float p0 = s[4 * g + e] > kEps ? s[4 * g + e] : 0.f;
                            if constexpr (DROP) {
                                const bool keep = lcg_keep(st_blk + (uint64_t)(8 * g + e) * row_step, thr);
                                s[4 * g + e] = keep ? p0 : 0.f;
                                xv[e] = keep ? p0 : -p0;
                            } else {
                                s[4 * g + e] = p0;
                                xv[e] = p0;
                            }
                        }
                        *reinterpret_cast<floatx4*>(xs + (g * 64 + lane) * 4) = xv;
                    }
                }
                __syncthreads();
                if (on) {
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const Bf3 pb = cut8([&](int i) { return s[8 * j + i]; });
#pragma unroll
                        for (int dt = 0; dt < DV / 32; ++dt)
                            dv[dt] = mfma_bf3<INF>(OT::tr(os + swO.tr0, os + swO.tr1, dt, 16 * j), pb, dv[dt]);
                    }
                }
                stage_next(qb, inf);
                __syncthreads();
            }
        };
        pass(std::false_type{});
        if (workgroup_any_nan<Cfg::NT / 64>(dv, tid)) pass(std::true_type{});
        if (key_ok && np > 1)
            store_rows_f32<DV, VEC>(p.part_dv + ((size_t)(part * B + b) * S_kv + my_k) * D_v, dv, 1.f, hh, D_v);
        else if (key_ok)
            store_rows_f32<DV, VEC>(static_cast<float*>(p.dv) + ((size_t)b * S_kv + my_k) * D_v, dv, p.c.keep_scale, hh, D_v);
    } else {
        // ----------------------------------------------------------- dS role
        Bf3 v[DV / 16];
        load_row_bf3<DV, VEC>(v, static_cast<const float*>(p.v) + (size_t)b * S_kv * D_v, my_k, S_kv, D_v, hh);
        const float ksc = p.c.keep_scale;
        floatx16 dk[DQK / 32];
        const DsLayout32 dsl(S_q, S_kv, causal);
        auto pass = [&](auto inf) {
            constexpr bool INF = decltype(inf)::value;
            if constexpr (INF) stage_first(inf);
#pragma unroll
            for (int dt = 0; dt < DQK / 32; ++dt) dk[dt] = floatx16{};
            __syncthreads();
            for (int qb = qb0; qb < nqb; ++qb) {
                const int q0 = qb * BQ;
                const uint32_t qs = (uint32_t)(((qb - qb0) & 1) * Cfg::STAGE), os = qs + (uint32_t)QT::BYTES;
                const bool on = live(q0);
                floatx16 dp = floatx16{};
                if (on) {
#pragma unroll
                    for (int ks = 0; ks < DV / 16; ++ks) dp = mfma_bf3<INF>(OT::row(os + swO.row, ks, 0), v[ks], dp);
                }
                stage_next(qb, inf);
                __syncthreads();
                if (on) {
                    // dS = P0 (keep ? dP / (1-p) : 0 - delta), P0 = |x|, keep = x > 0
                    const float* Fs = reinterpret_cast<const float*>(smem + os + OT::BYTES);
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const floatx4 xv = *reinterpret_cast<const floatx4*>(xs + (g * 64 + lane) * 4);
                        const floatx4 de4 = *reinterpret_cast<const floatx4*>(Fs + BQ + 8 * g + 4 * hh);
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            float d = DROP ? dp[4 * g + e] * ksc : dp[4 * g + e];
                            float p0 = xv[e];
                            if constexpr (DROP) {
                                d = xv[e] > 0.f ? d : 0.f;
                                p0 = __builtin_fabsf(xv[e]);
                            }
                            dp[4 * g + e] = p0 * (d - de4[e]);
                        }
                    }
                    if constexpr (DS) {
                        // the lane's 16 values as four 16-byte slots of its key
                        // group (DsLayout32), each store 1 KB whole, non-temporal;
                        // zero for keys past S_kv (dQ reads them unmasked)
                        unsigned char* grp = static_cast<unsigned char*>(p.ds) + dsl.offset(b, kt, qb) + kw * 4096;
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            floatx4 x;
#pragma unroll
                            for (int e = 0; e < 4; ++e) x[e] = key_ok ? dp[4 * u + e] : 0.f;
                            __builtin_nontemporal_store(
                                x, reinterpret_cast<floatx4*>(grp + DsLayout32::slot32(l32, 16 * hh + 4 * u)));
                        }
                    }
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const Bf3 db = cut8<INF>([&](int i) { return dp[8 * j + i]; });
#pragma unroll
                        for (int dt = 0; dt < DQK / 32; ++dt)
                            dk[dt] = mfma_bf3<INF>(QT::tr(qs + swQ.tr0, qs + swQ.tr1, dt, 16 * j), db, dk[dt]);
                    }
                }
                __syncthreads();
            }
        };
        pass(std::false_type{});
        if (workgroup_any_nan<Cfg::NT / 64>(dk, tid)) pass(std::true_type{});
        if (key_ok && np > 1)
            store_rows_f32<DQK, VEC>(p.part_dk + ((size_t)(part * B + b) * S_kv + my_k) * D_qk, dk, 1.f, hh, D_qk);
        else if (key_ok)
            store_rows_f32<DQK, VEC>(static_cast<float*>(p.dk) + ((size_t)b * S_kv + my_k) * D_qk, dk, p.c.scale, hh, D_qk);
    }
}

}  // namespace

hipError_t launch_bwd_dkdv_f32(const BwdParams& p, bool vec, hipStream_t stream) {
    const int B = p.s.B, S_kv = p.s.S_kv;
    if (B == 0 || S_kv == 0) return hipSuccess;
    if (fp32_chain(p.s)) return launch_bwd_dkdv_f32_chain(p, vec, stream);
    return with_dim(p.s.D_qk, [&](auto dqk) {
        return with_dim(p.s.D_v, [&](auto dv) {
            return with_bool(vec, [&](auto v) {
                return with_bool(p.c.use_dropout != 0, [&](auto d) {
                    constexpr int DQK = decltype(dqk)::value, DV = decltype(dv)::value;
                    constexpr bool V = decltype(v)::value, D = decltype(d)::value;
                    using Cfg = DkvBf3Cfg<DQK, DV>;
                    static_assert(Cfg::BKV == DsLayout32::KT && Cfg::BQ == DsLayout32::QBK, "dS chunk geometry");
                    const dim3 n = tile_grid((long long)((S_kv + Cfg::BKV - 1) / Cfg::BKV) * p.kv_parts * B, Cfg::NT);
                    const int win = row_window((size_t)p.s.S_q * (DQK + DV) * 4);
                    if constexpr (V && (DQK == 128 || DV == 128)) {
                        if (p.ds)
                            return launch_kernel<sdpa_bwd_dkdv_f32_bf3_kernel<DQK, DV, V, D, true>>(n, Cfg::NT, Cfg::LDS_BYTES,
                                                                                               stream, p, win);
                    }
                    if (p.ds) return hipErrorInvalidValue;  // the dS path's shapes are aligned, with a 128-wide side
                    return launch_kernel<sdpa_bwd_dkdv_f32_bf3_kernel<DQK, DV, V, D, false>>(n, Cfg::NT, Cfg::LDS_BYTES,
                                                                                        stream, p, win);
                });
            });
        });
    });
}

}  // namespace sdpa
