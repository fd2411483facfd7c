// sdpa_parts.h -- which forward a shape runs where the query side has few
// tiles, and how the streamed side of a tile is divided over workgroups.
#pragma once

#include <stddef.h>

#include <hip/hip_runtime.h>

namespace sdpa {

// First of n blocks in part `part` of np (equal lengths, +-1).
__host__ __device__ inline int part_begin(int n, int part, int np) { return (int)((long long)n * part / np); }

// Tile height and waves of the kernels for small grids.
constexpr int kSmallRows = 32, kSmallWaves = 4;

struct FwdPlan {
    bool small;             // the kernel for small grids
    int parts;              // workgroups that share a tile's keys (merged by a second kernel)
    size_t o_bytes, bytes;  // workspace of the parts' O, and in all (0 with one part)
};

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
    if (!f16 || B <= 0 || S_q <= 0) return f;
    const auto pad = [](int d) { return d <= 32 ? 32 : (d <= 64 ? 64 : 128); };
    const long long tiles = (long long)B * ((S_q + kSmallRows - 1) / kSmallRows);
    const long long slots = pad(D_qk) + pad(D_v) <= 160 ? 512 : 256;
    f.small = tiles <= (causal && S_q >= 1000 ? 2 * slots : slots);
    if (!f.small || causal || tiles > slots / 2) return f;
    const long long blocks = ((long long)S_kv + kSmallRows - 1) / kSmallRows;
    const long long walk = (blocks + kSmallWaves - 1) / kSmallWaves;  // blocks per wave, undivided
    long long n = 256 / tiles;
    if (slots == 512 && (n < 1 || walk / n >= 12)) n = slots / tiles;
    if (n > walk / 2) n = walk / 2;
    if (n < 2 || walk - walk / n < 9) return f;
    f.parts = (int)n;
    const size_t rows = (size_t)f.parts * B * S_q;
    f.o_bytes = (rows * D_v * 4 + 255) & ~(size_t)255;
    f.bytes = f.o_bytes + rows * 8;
    return f;
}

}  // namespace sdpa
