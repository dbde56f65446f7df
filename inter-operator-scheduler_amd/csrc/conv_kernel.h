// The stand-alone kernel around a convolution body.
#pragma once

#include <climits>
#include <cstddef>

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

// Several convolutions of one input, with the same window, on one body: grid = the tiles of all members, their tiles of channels one
// behind the other, so that the blocks of an XCD that read a tile of pixels run together.  A block finds its member from the
// kernel-argument segment.
// A staged block is a chain of loads, conversions, barriers and matrix work that nothing but another block on its compute unit covers:
// alone, 64 x 64 tiles of 768 -> 192 channels on 17 x 17 take 16 us at batch 3 as at batch 7.  Four such convolutions together put three to
// seven blocks on a compute unit instead of one or two: 27 -> 12 us (half, batch 7), 41 -> 19 us (bfloat16, batch 16), 133 -> 99 us (fp32, batch 64: 606
// TFLOP/s of half products).
// Six of the two-term kernels (64 x 128 and 128 x 64 outputs) keep 16 bytes a lane in scratch memory over the sums' tests: two stores and
// two loads per tile behind its K loop, for the fourth wavefront on a SIMD.
struct ConvBatchArgs {
    int xcd_q, xcd_r, tile_div, weights_major;   // as in ConvKernelArgs, of all members' tiles
    FastDiv div_tile;
    int first[kMaxConvBatch];                    // first tile of channels of a member (INT_MAX: there is none)
    ConvKernelArgs item[kMaxConvBatch];          // (numbered by rows of tiles of channels, without XCDs)
};
typedef void (*ConvBatchKernelFn)(ConvBatchArgs);
extern const ConvBatchKernelFn kPipeBatchKernels[][2];   // conv_batch.hip, in the order of conv_pipe.h; [1]: all members PLAIN
template <typename Body>
__global__ __launch_bounds__(Body::THREADS) __attribute__((amdgpu_waves_per_eu(waves_per_simd<Body>::value))) void conv_batch_kernel(ConvBatchArgs b) {
    extern __shared__ floatx4 conv_smem[];
    const int xcd = blockIdx.x & 7, t = (int)(blockIdx.x >> 3) + xcd * b.xcd_q + min(xcd, b.xcd_r);
    const int q = (int)fast_div((unsigned)t, b.div_tile), rest = t - q * b.tile_div;
    const int m = b.weights_major ? q : rest, n = b.weights_major ? rest : q;
    int i = 0, first = 0;
#pragma unroll
    for (int k = 1; k < kMaxConvBatch; k++) {
        i += m >= b.first[k] ? 1 : 0;
        first = m >= b.first[k] ? b.first[k] : first;
    }
    // (read in place, through the segment's address: indexing the by-value parameter costs registers)
    typedef const ConvKernelArgs __attribute__((address_space(4))) *ConstantArgs;
    unsigned long long address = (unsigned long long)__builtin_amdgcn_kernarg_segment_ptr() + offsetof(ConvBatchArgs, item);
    asm volatile("" : "+s"(address));
    address += (unsigned)__builtin_amdgcn_readfirstlane(i) * (unsigned)sizeof(ConvKernelArgs);
    const ConvKernelArgs &a = *(const ConvKernelArgs *)(ConstantArgs)address;
    Body::template run<false>(a, reinterpret_cast<float *>(conv_smem), __builtin_amdgcn_readfirstlane(n * a.tiles_m + m - first) << 3, 0, 0);
}

}  // namespace ios
