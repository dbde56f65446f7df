// The stand-alone kernel around a convolution body.
#pragma once

#include "conv_body.h"

namespace ios {

// stand-alone kernel around a body: grid = (tiles, groups, K slices), dynamic LDS = Body::SMEM_FLOATS floats
// RES: the residual form of the epilogue (a.res is not null)
template <typename Body, bool RES = false>
__global__ __launch_bounds__(Body::THREADS) void conv_kernel(ConvKernelArgs a) {
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
