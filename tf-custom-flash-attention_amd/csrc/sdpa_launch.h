// sdpa_launch.h -- host-side launch helpers shared by the forward and backward
// launchers: compile-time dispatch over the padded feature widths and flags,
// and a launch wrapper that raises the dynamic-LDS limit once per kernel.
#pragma once

#include <hip/hip_runtime.h>

#include <mutex>
#include <type_traits>

#include "sdpa_params.h"

namespace sdpa {

enum class DType : int { F32 = 0, F16 = 1 };

// Padded feature width for D in [0, 128]: the MFMA tiles are 32 wide in the
// output direction, so every kernel is instantiated for 32, 64 and 128
// (the reference buckets max(D_qk, D_v) into 8/16/32/64/128,
// sdpa/sdpa_fwd.cu.cc:191-215; here D_qk and D_v are bucketed separately).
template <typename F>
hipError_t with_dim(int d, F&& f) {
    if (d <= 32) return f(std::integral_constant<int, 32>{});
    if (d <= 64) return f(std::integral_constant<int, 64>{});
    return f(std::integral_constant<int, 128>{});
}

template <typename F>
hipError_t with_bool(bool b, F&& f) {
    if (b) return f(std::true_type{});
    return f(std::false_type{});
}

// Grid of n workgroups: one dimension, or rows of 2^22 where that would pass
// the 2^32 - 1 threads HIP launches per dimension (tiles of 512 threads: 2^23
// batch rows of up to 128 queries).  The kernel takes tile_id() and leaves
// where it is n or more.
inline dim3 tile_grid(long long n, unsigned block) {
    if (n * block <= 0xFFFFFFFFll) return dim3((unsigned)n);
    return dim3(1u << 22, (unsigned)((n + (1 << 22) - 1) >> 22));
}
__device__ __forceinline__ int tile_id() { return (int)(blockIdx.x + gridDim.x * blockIdx.y); }

// Launch `kern` with `lds` bytes of dynamic LDS.  The per-kernel attribute is
// set once per process (gfx950 has 160 KB of LDS per CU; kernels here use up
// to all of it, which each checks).
// The kernel is a template argument so that each kernel gets its own once-flag.
template <auto kern, typename... Args>
hipError_t launch_kernel(dim3 grid, unsigned block, size_t lds, hipStream_t stream,
                         const Args&... args) {
    static std::once_flag once;
    static hipError_t attr_err = hipSuccess;
    std::call_once(once, [&] {
        attr_err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    });
    if (attr_err != hipSuccess) return attr_err;
    if (grid.x == 0) return hipSuccess;
    if ((unsigned long long)grid.x * block > 0xFFFFFFFFull) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL(kern, grid, dim3(block), lds, stream, args...);
    return hipGetLastError();
}

// fp16 forward for any D and alignment (sdpa_fwd.hip)
hipError_t launch_fwd_f16(const FwdParams& p, bool vec, hipStream_t stream);
// fp32 forward on the bf16 matrix cores (sdpa_f32_fwd.hip)
hipError_t launch_fwd_f32(const FwdParams& p, bool vec, hipStream_t stream);
// phases: kBwdDq (dQ kernel, writes delta) and/or kBwdDkDv (reads delta).
constexpr int kBwdDq = 1, kBwdDkDv = 2;
// half4: fp16 rows of a multiple of 4 features that the kernels for small
// grids take.
hipError_t launch_bwd(const BwdParams& p, DType dtype, bool vec, bool half4, int phases, hipStream_t stream);

// fp16 kernels fed by HBM -> LDS copies (sdpa_f16_fwd.hip, sdpa_f16_dq.hip,
// sdpa_f16_dkdv.hip).  They require D_qk and D_v to be multiples of 8 and
// every tensor 16-byte aligned.
hipError_t launch_fwd_f16_dma(const FwdParams& p, hipStream_t stream);
// The same for grids too small to fill the chip (sdpa_f16_fwd_small.hip);
// p.parts and the part buffers as planned by fwd_plan().
hipError_t launch_fwd_f16_wave(const FwdParams& p, hipStream_t stream);
hipError_t launch_bwd_f16_dma(const BwdParams& p, int phases, hipStream_t stream);
// dQ phase of launch_bwd_f16_dma (sdpa_f16_dq.hip)
hipError_t launch_bwd_dq_f16_dma(const BwdParams& p, hipStream_t stream);
// dK/dV phase of launch_bwd_f16_dma at a 128-wide side (D_qk or D_v = 128;
// sdpa_f16_dkdv_split.hip); with p.ds set it also stores dS' (DsLayout)
hipError_t launch_bwd_dkdv_f16_split(const BwdParams& p, hipStream_t stream);

// dS path of the fp16 DMA backward (sdpa_f16_dq_ds.hip), for the shapes the
// split dK/dV kernels serve: the row values (stats2, delta), then
// launch_bwd_dkdv_f16_split with p.ds, then dQ from the stored dS'.
inline bool bwd_ds_shape(int D_qk, int D_v) { return D_qk > 64 || D_v > 64; }
hipError_t launch_bwd_rows_f16(const BwdParams& p, hipStream_t stream);
hipError_t launch_bwd_dq_ds_f16(const BwdParams& p, hipStream_t stream);
// The same three kernels, and dQ of the other path, for grids too small to
// fill the chip (sdpa_f16_bwd_small.hip); p.parts as planned.
hipError_t launch_bwd_dq_f16_wave(const BwdParams& p, hipStream_t stream);
hipError_t launch_bwd_dkdv_f16_wave(const BwdParams& p, hipStream_t stream);
hipError_t launch_bwd_dq_ds_f16_wave(const BwdParams& p, hipStream_t stream);
// The same path for fp32 (sdpa_f32_dq_ds.hip, sdpa_f32_dkdv.hip).
// fp32 dQ of the path without stored dS at D <= 64, on the bf16 matrix cores,
// and the sums of the parts where p.parts or p.kv_parts are more than one
// (sdpa_f32_dq.hip)
hipError_t launch_bwd_dq_f32(const BwdParams& p, bool vec, hipStream_t stream);
hipError_t launch_bwd_merge_f32(const BwdParams& p, hipStream_t stream);
// fp32 dK/dV on the bf16 matrix cores (sdpa_f32_dkdv.hip); with p.ds set it
// also stores dS
hipError_t launch_bwd_dkdv_f32(const BwdParams& p, bool vec, hipStream_t stream);
hipError_t launch_bwd_rows_f32(const BwdParams& p, hipStream_t stream);
hipError_t launch_bwd_dq_ds_f32(const BwdParams& p, hipStream_t stream);

// The fp32 forward of the shapes of fp32_chain_fwd() and dK/dV of those of
// fp32_chain() (sdpa_f32_chain.hip).
hipError_t launch_fwd_f32_chain(const FwdParams& p, bool vec, hipStream_t stream);
hipError_t launch_bwd_dkdv_f32_chain(const BwdParams& p, bool vec, hipStream_t stream);

}  // namespace sdpa
