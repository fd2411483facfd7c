// sdpa_parts.h -- which forward a shape runs where the query side has few
// tiles, and how the streamed side of a tile is divided over workgroups.
#pragma once

#include <stddef.h>

#include <hip/hip_runtime.h>

#include "sdpa_params.h"

namespace sdpa {

// First of n blocks in part `part` of np (equal lengths, +-1).
__host__ __device__ inline int part_begin(int n, int part, int np) { return (int)((long long)n * part / np); }

// Tile height and waves of the kernels for small grids.
constexpr int kSmallRows = 32, kSmallWaves = 4;

// fp16 feature sizes (multiples of 4 up to 64) that the kernels for small
// grids take and the copies of whole 16-byte chunks do not (sdpa_wave.h, keep4).
inline bool half4_dims(int D_qk, int D_v) {
    return D_qk > 0 && D_v > 0 && D_qk % 4 == 0 && D_v % 4 == 0 && D_qk <= 64 && D_v <= 64 &&
           !(D_qk % 8 == 0 && D_v % 8 == 0);
}

struct FwdPlan {
    bool small;             // the kernel for small grids
    int parts;              // workgroups that share a tile's keys (merged by a second kernel)
    size_t o_bytes, bytes;  // workspace of the parts' O, and in all (0 with one part)
};

// The number of parts with the least estimated time for `tiles` tiles of
// `blocks` streamed blocks each on 256 workgroups at a time (one per CU):
// block_us per block, 4 us per workgroup besides, and with several parts the
// second kernel, merge_us and its traffic (part_bytes per part, written and
// read, at 2.5 TB/s).  Under the causal mask a tile has half of the blocks
// on average, one of them all.
inline int least_time_parts(long long tiles, long long blocks, bool causal, double block_us, double merge_us,
                            double part_bytes, int slots = 256) {
    if (tiles > slots || blocks < 2) return 1;
    int best = 1;
    double best_us = 0;
    for (int n = 1; n <= blocks && n <= 64; ++n) {
        const double chain = 4 + (double)((blocks + n - 1) / n) * block_us;
        double us = (double)((tiles * n + slots - 1) / slots) * chain;
        if (causal) {
            const double work = (double)tiles * (4 * n + 0.5 * blocks * block_us) / slots + chain / 2;
            us = work > chain ? work : chain;
        }
        if (n > 1) us += merge_us + n * part_bytes / 2.5e6;
        if (n == 1 || us < 0.95 * best_us) {
            best = n;
            best_us = us;
        }
    }
    return best;
}

inline int pad_dim(int d) { return d <= 32 ? 32 : (d <= 64 ? 64 : 128); }

// fp32 shapes that keep the sequential fp32 sums of sdpa_f32_chain.hip, where
// the gate of the gradient lies among the weights of ordinary rows (figures
// there: none of 40 calls differed up to 12000 keys, 11 of 38 at 16384; for
// scores of unit variance the weights near the gate grow 16-fold from 8192 to
// 16384 keys).  The gradient's kernels go by the keys alone: given q, k and
// stats, a weight keeps its side.  The forward of up to 16 queries (generation)
// divides its keys on the bf16 matrix cores; its stats, 2e-6 from the chain's
// at most, moved a weight in 0, 2 and 11 of 20 calls at B 64, S_q 16, S_kv
// 16384, D 64 and 128, and S_q 4, S_kv 32768 (with the gradient there as well
// 3, 7 and 20; the largest change of an element 7e-4 of the root mean square).
inline bool fp32_chain(const AttnShape& s) { return s.S_kv > 8192; }
// The forward also where few keys meet more than 256 tiles of 128 queries: two
// of its workgroups of four waves share a CU and start sooner than one of
// eight, and its blocks are of 32 keys.  Chain -> bf16 parts, us: B 100, S_q
// 1000, D 64, 8 keys 23.4 -> 37.0, 64 keys 31.8 -> 39.0, 129 keys 56.7 -> 58.3,
// 192 keys 65.6 -> 61.1; D 32, 129 keys 33.4 -> 39.0, 192 keys 37.2 -> 39.4, 256
// keys 47.1 -> 45.9; B 600, causal, D 128, S 129 97 -> 117, S 192 126 -> 132.
inline bool fp32_chain_fwd(const AttnShape& s, bool causal) {
    const int few = causal || (s.D_qk <= 32 && s.D_v <= 32) ? 192 : 160;
    const long long tiles = (long long)s.B * ((s.S_q + 127) / 128);
    if (s.S_kv <= few && tiles > 256 && tiles < 1 << 24) return true;  // (its grid has one dimension)
    return fp32_chain(s) && s.S_q > 16;
}

// Parts of the keys of a 128-query tile in the fp32 forward (sdpa_f32_fwd.hip).
// A block (64 keys, 32 where both sides are 128 wide) takes about 0.0215 us
// per padded feature column of K and V: 2.35 measured at 64 + 64, 4.2 at 128
// + 64, 2.95 for 32 keys at 128 + 128.  Undivided -> chosen, us: B 8, S_q 1,
// S_kv 8000, D 64: 288 -> 22.6 (32 parts); B 64, S_q 64, S_kv 2000, D 128:
// 194 -> 65 (4); B 24, S 700, D 64: 38 (1; in two parts 57: a second round).
inline int fwd_f32_parts(int B, int S_q, int S_kv, int D_qk, int D_v, bool causal) {
    if (fp32_chain_fwd(AttnShape{B, S_q, S_kv, D_qk, D_v}, causal)) return 1;
    const int pq = pad_dim(D_qk), pv = pad_dim(D_v);
    const bool wide = pq == 128 && pv == 128;
    return least_time_parts((long long)B * ((S_q + 127) / 128), ((long long)S_kv + (wide ? 31 : 63)) / (wide ? 32 : 64),
                            causal, wide ? 2.95 : 0.0215 * (pq + pv), 4, 8.0 * B * S_q * D_v);
}

// The fp16 forward of a shape, from its count of 32-query tiles (all times
// in us, 128-query kernel -> 32-query kernel).
//
// The 32-query kernel wins while its workgroups are all resident at once:
// one per CU at a 128-wide side, two where both padded widths sum to at most
// 160 (its LDS ring).  At D = 64: 512 tiles 13.1 -> 8.7 (B 32, S 512,
// causal), 1024 tiles 13.8 -> 14.6 (B 64).  At D = 128: 256 tiles 16.0 ->
// 11.5 (B 16, S 512, causal), 512 tiles 16.6 -> 19.0 (B 32).  A long causal
// side keeps the 128-query kernel waiting for its heaviest tiles, so there
// the line lies at two rounds: 44 -> 31 (B 8, S 2048, D 128: 512 tiles),
// 36 -> 28 (B 16, S 2048, D 64: 1024 tiles), 44 -> 58 (B 16, D 128: 1024).
//
// A tile's keys are divided once each wave would walk so many 32-key blocks
// that the division saves more than the merge kernel costs (about 5 us, nine
// blocks): into as many parts as give 256 workgroups, or 512 where two share
// a CU and a dozen blocks would remain per wave, but at least two blocks a
// wave.  B 64, S_q 1, S_kv 4096, D 128: 68 -> 36.8 in one part, 27.7 in
// four (134 MB); B 16, S_q 64, S_kv 8192, D 64: 112 -> 46.6, 16.1 in eight;
// B 128, S_q 1, S_kv 1000, D 128: 14.5 in one, 18.7 in two.
inline FwdPlan fwd_plan(bool f16, int B, int S_q, int S_kv, int D_qk, int D_v, bool causal) {
    FwdPlan f{false, 1, 0, 0};
    // (without values there is only stats to write, which the small kernel and
    // the merge kernel write with a row's first columns)
    if (B <= 0 || S_q <= 0 || D_v == 0) return f;
    // fp16 widths that the register-staged kernel serves, which divides
    // nothing; with rows of half chunks only the 32-query kernel divides
    const bool chunks = D_qk % 8 == 0 && D_v % 8 == 0;
    if (f16 && !chunks && !half4_dims(D_qk, D_v)) return f;
    const auto divide = [&](long long n) {
        if (f16 && !f.small && !chunks) return;
        f.parts = (int)n;
        const size_t rows = (size_t)f.parts * B * S_q;
        f.o_bytes = (rows * D_v * 4 + 255) & ~(size_t)255;
        f.bytes = f.o_bytes + rows * 8;
    };
    if (!f16) {
        divide(fwd_f32_parts(B, S_q, S_kv, D_qk, D_v, causal));
        if (f.parts == 1) f.o_bytes = f.bytes = 0;
        return f;
    }
    const long long tiles = (long long)B * ((S_q + kSmallRows - 1) / kSmallRows);
    const long long slots = pad_dim(D_qk) + pad_dim(D_v) <= 160 ? 512 : 256;
    f.small = tiles <= (causal && S_q >= 1000 ? 2 * slots : slots);
    const long long blocks = ((long long)S_kv + kSmallRows - 1) / kSmallRows;
    const long long walk = (blocks + kSmallWaves - 1) / kSmallWaves;  // blocks per wave, undivided
    // The 128-query kernel with its keys divided, 512 workgroups at a time:
    // where the 32-query one does not run, or has no workgroup to spare for a
    // division and a longer walk (a block there takes 0.65 us, 1.05 at a
    // 128-wide side).  B 32, S_q 300, S_kv 2000, D 128: 43 -> 33 (3 parts);
    // B 32, S_q 400, S_kv 8000, D 128: 145 -> 81 (4); B 64, S_q 300, S_kv
    // 1500, D 80: 39.9, in two parts 39.3.
    if (!causal && (!f.small || tiles > slots / 2)) {
        const long long big = (long long)B * ((S_q + 127) / 128), steps = ((long long)S_kv + 63) / 64;
        const int n = least_time_parts(big, steps, false, 1.25, 8, 8.0 * B * S_q * D_v, 512);
        const double big_us = 12 + (double)((steps + n - 1) / n) * 1.25 + n * 8.0 * B * S_q * D_v / 2.5e6;
        if (n > 1 && (!f.small || big_us < 4 + walk * (slots == 512 ? 0.65 : 1.05))) {
            f.small = false;
            divide(n);
            return f;
        }
    }
    if (!f.small || causal || tiles > slots / 2) return f;
    long long n = 256 / tiles;
    if (slots == 512 && (n < 1 || walk / n >= 12)) n = slots / tiles;
    if (n > walk / 2) n = walk / 2;
    if (n < 2 || walk - walk / n < 9) return f;
    divide(n);
    return f;
}

// ---- backward: where the kernels of sdpa_f16_bwd_small.hip run (times of
// the whole backward in us, large kernel -> small kernel, dropout 0.1 where
// S_q = S_kv).  As in the forward a small kernel wins while its workgroups
// are resident at once, and under the causal mask, where the large kernels
// wait for their heaviest tiles, up to twice that on long sides.
inline long long small_tiles(int B, int S, int rows) { return (long long)B * ((S + rows - 1) / rows); }

// dQ at D <= 64, two workgroups per CU.  512 tiles: 36.6 -> 32.4 (B 32, S
// 512, causal), 61.5 -> 56.5 (B 16, S 1000); 1024 tiles: 37.5 -> 40.6 (B 64,
// S 512, causal) but 111 -> 103 (B 16, S 2048, causal).
inline bool dq_small(const AttnShape& s, bool causal) {
    if (s.D_qk > 64 || s.D_v > 64) return false;
    return small_tiles(s.B, s.S_q, kSmallRows) <= (causal && s.S_q >= 1000 ? 1024 : 512);
}

// Workgroups that share a tile's keys in that kernel: as many as give 256
// workgroups (512 where a dozen blocks would remain per wave), at least two
// blocks a wave, where it saves each wave at least six blocks (about what the
// merge kernel costs).  B 16, S_q 64, S_kv 4000: 40.3 in one part, 23.7 in
// eight; B 64, S_q 64, S_kv 1000: 23.6 in one, 23.9 in two.
inline int dq_parts(const AttnShape& s, bool causal) {
    if (causal || !dq_small(s, causal) || s.B <= 0 || s.S_q <= 0) return 1;
    const long long tiles = small_tiles(s.B, s.S_q, kSmallRows);
    const long long walk = (small_tiles(1, s.S_kv, kSmallRows) + kSmallWaves - 1) / kSmallWaves;
    long long n = 256 / tiles;
    if (n < 1 || walk / n >= 12) n = 512 / tiles;
    if (n > walk / 2) n = walk / 2;
    return n < 2 || walk - walk / n < 6 ? 1 : (int)n;
}

// dK/dV, two workgroups per CU up to D = 64, one at a 128-wide side.  Each of
// the four waves needs a query block of its own to win.  D = 64: 512 tiles
// 23.9 -> 19.2 (B 64, S 256, causal), 1024 tiles 25.2 -> 26.3 (B 128, S 256)
// but 62.1 -> 48.2 (B 32, S 1000, causal), 2048 tiles 66.6 -> 70.3 (B 64).
// D = 128: 256 tiles 46.8 -> 39.6 (B 16, S 512, causal), 512 tiles 48.2 ->
// 51.5 (B 32, S 512) but 77.2 -> 69.9 (B 16, S 1000, causal).  S_q 16,
// S_kv 4000, B 4, D 64: 62.3 -> 64.2.
inline bool dkdv_small(const AttnShape& s, bool causal) {
    if (s.S_q <= 3 * kSmallRows) return false;
    const long long tiles = small_tiles(s.B, s.S_kv, kSmallRows);
    if (s.D_qk > 64 || s.D_v > 64) return tiles <= (causal && s.S_q >= 1000 ? 512 : 256);
    return tiles <= (s.S_q >= 512 ? 1024 : 512);
}

// dQ from the stored dS', 64-query tiles, one workgroup per CU: two rounds of
// them still win, as the large kernel's tiles are four times as high.  512
// tiles: 51.7 -> 45.1 (B 64, S 512, D 128, causal), 83.6 -> 77.9 (B 32, S
// 1000); 1024 tiles: 141 -> 150 (B 64, S 1000) but 161 -> 147 (B 32, S 2048,
// causal).  B 16, S_q 64, S_kv 4000: 115 -> 56.
inline bool dq_ds_small(const AttnShape& s, bool causal) {
    return small_tiles(s.B, s.S_q, 64) <= (causal && s.S_q >= 1000 ? 1024 : 512);
}

// Workgroups that share a tile in the backward of a shape without a dS path
// (D <= 64), and the floats of workspace their sums take: dQ tiles divided
// over keys, fp32 also dK/dV tiles over queries.
struct BwdParts {
    int q, kv;
    size_t dq_floats, dk_floats, dv_floats;
    size_t floats() const { return dq_floats + dk_floats + dv_floats; }
};

inline BwdParts bwd_parts(bool f16, const AttnShape& s, bool causal) {
    BwdParts r{1, 1, 0, 0, 0};
    if (s.D_qk > 64 || s.D_v > 64 || s.B <= 0 || s.S_q <= 0 || s.S_kv <= 0) return r;
    if (f16) {
        // (the register-staged kernel of other widths divides nothing)
        if ((s.D_qk % 8 == 0 && s.D_v % 8 == 0) || half4_dims(s.D_qk, s.D_v)) r.q = dq_parts(s, causal);
    } else if (!fp32_chain(s)) {
        // Blocks of 64 keys (dQ, 3.25 us measured at D = 64) and of 32 queries
        // (dK/dV, 1.9).  Undivided -> chosen, us of the whole backward: B 8,
        // S_q 64, S_kv 8000, D 64: 453 -> 94 (8 parts of dQ; more now); B 8,
        // S 700, causal, D 64: 110 -> 80 (4 of dK/dV alone); B 20, S 400, D
        // 32/4: 49.4 -> 41.5 (2 of dK/dV); B 64, S 512, causal: 100, undivided
        // (in two parts of dQ 113).
        const double cols = pad_dim(s.D_qk) + pad_dim(s.D_v);
        r.q = least_time_parts((long long)s.B * ((s.S_q + 127) / 128), ((long long)s.S_kv + 63) / 64, causal,
                               1.0 + 0.0175 * cols, 3, 8.0 * s.B * s.S_q * s.D_qk);
        r.kv = least_time_parts((long long)s.B * ((s.S_kv + 127) / 128), ((long long)s.S_q + 31) / 32, causal,
                                0.8 + 0.0085 * cols, 3, 8.0 * s.B * s.S_kv * (s.D_qk + s.D_v));
    }
    if (!f16 && fp32_chain(s) && s.S_q <= 16)
        // Blocks of 32 keys of the sequential sums (3.5 us at D = 64), for the
        // few queries whose forward divides too; the gate does not see the
        // division.  Undivided -> chosen, us of the whole backward at D = 64: B
        // 64, S_q 16, S_kv 16384: 2237 -> 866; B 16, S_q 8, S_kv 12000: 1468 ->
        // 177; B 1, S_q 16, S_kv 65536: 7299 -> 164 (on the bf16 matrix cores
        // 536, 113 and 91).
        r.q = least_time_parts(s.B, ((long long)s.S_kv + 31) / 32, causal,
                               0.036 * (pad_dim(s.D_qk) + 0.5 * pad_dim(s.D_v)), 3, 8.0 * s.B * s.S_q * s.D_qk);
    if (r.q > 1) r.dq_floats = (size_t)r.q * s.B * s.S_q * s.D_qk;
    if (r.kv > 1) {
        r.dk_floats = (size_t)r.kv * s.B * s.S_kv * s.D_qk;
        r.dv_floats = (size_t)r.kv * s.B * s.S_kv * s.D_v;
    }
    return r;
}

}  // namespace sdpa
