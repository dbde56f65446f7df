// The stand-alone kernel around a convolution body.
#pragma once

#include "conv_body.h"

namespace ios {

// Wavefronts per SIMD that a body's registers must leave room for (what its block takes, where the body names no number): left to
// itself the compiler gives accumulators that leave a loop a second set of registers.
template <typename Body, typename = void>
struct waves_per_simd { static constexpr int value = (Body::THREADS + 255) / 256; };
template <typename Body>
struct waves_per_simd<Body, std::void_t<decltype(Body::WAVES_PER_SIMD)>> {
    static constexpr int value = Body::WAVES_PER_SIMD > (Body::THREADS + 255) / 256 ? Body::WAVES_PER_SIMD : (Body::THREADS + 255) / 256;
};

// stand-alone kernel around a body: grid = (tiles, groups, K slices), dynamic LDS = Body::SMEM_FLOATS floats
// RES: the residual form of the epilogue (a.res is not null)
template <typename Body, bool RES = false>
__global__ __launch_bounds__(Body::THREADS) __attribute__((amdgpu_waves_per_eu(waves_per_simd<Body>::value))) void conv_kernel(ConvKernelArgs a) {
    extern __shared__ floatx4 conv_smem[];
    if (a.xcd_local) {   // one-dimensional grid numbered for split-K inside an XCD
        const XcdSlot slot = xcd_enter(a, blockIdx.x, blockIdx.x);
        if (slot.idle) return;
        Body::template run<RES>(a, reinterpret_cast<float *>(conv_smem), slot.tile, 0, slot.slice);
        return;
    }
    Body::template run<RES>(a, reinterpret_cast<float *>(conv_smem), blockIdx.x, blockIdx.y, blockIdx.z);
}

}  // namespace ios
