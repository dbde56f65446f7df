// Convolutions of different inputs and windows, and a pool, in a launch.
#pragma once

#include "conv_kernel.h"
#include "pointwise_body.h"

namespace ios {

// On one body: the blocks of one member behind those of the other, each member numbered over the XCDs by itself (first: a multiple of eight;
// the blocks between two members have no tile), and those of the pool behind all.
// What a level of parallel branches holds, 1 x 7 beside 7 x 1 on 17 x 17, is a third to a whole round of blocks each, and a staged block alone on
// its compute unit waits for its own loads, barriers and matrix work: at batch 16 20.4 us for one of them (192 channels), 20.0 for both.
// The pool is bound by memory and takes what they leave.
struct ConvMixedArgs {
    int first[kMaxConvBatch];                    // first block of a member (INT_MAX: there is none)
    int pool_first, pool_blocks;                 // (INT_MAX, 0: there is none)
    PoolArgs pool;
    ConvKernelArgs item[kMaxConvBatch];
};
typedef void (*ConvMixedKernelFn)(ConvMixedArgs);
// conv_mixed.hip, in the order of conv_pipe.h ([1]: all members PLAIN) and conv_window.h
extern const ConvMixedKernelFn kPipeMixedKernels[][2], kWindowMixedKernels[];
extern const ConvMixedKernelFn kWindow7MixedKernels[], kWindow9MixedKernels[];   // conv_mixed7.hip, conv_mixed9.hip
// (Where four wavefronts a SIMD fit, the address of the member's arguments is one value too many.)
template <typename Body>
struct mixed_waves { static constexpr int value = waves_per_simd<Body>::value == 4 ? 3 : waves_per_simd<Body>::value; };
template <typename Body>
__global__ __launch_bounds__(Body::THREADS) __attribute__((amdgpu_waves_per_eu(mixed_waves<Body>::value))) void conv_mixed_kernel(ConvMixedArgs b) {
    extern __shared__ floatx4 conv_smem[];
    // (read in place, as in conv_batch_kernel)
    typedef const __attribute__((address_space(4))) char *ConstantBytes;
    ConstantBytes segment = (ConstantBytes)__builtin_amdgcn_kernarg_segment_ptr();
    if ((int)blockIdx.x >= b.pool_first) {
        const PoolArgs &pool = *(const PoolArgs *)(const PoolArgs __attribute__((address_space(4))) *)(segment + offsetof(ConvMixedArgs, pool));
        pool_body(pool, (int)blockIdx.x - b.pool_first, b.pool_blocks, Body::THREADS);
        return;
    }
    int i = 0, first = 0;
#pragma unroll
    for (int k = 1; k < kMaxConvBatch; k++) {
        i += (int)blockIdx.x >= b.first[k] ? 1 : 0;
        first = (int)blockIdx.x >= b.first[k] ? b.first[k] : first;
    }
    unsigned long long address = (unsigned long long)segment + offsetof(ConvMixedArgs, item);
    asm volatile("" : "+s"(address));
    address += (unsigned)__builtin_amdgcn_readfirstlane(i) * (unsigned)sizeof(ConvKernelArgs);
    const ConvKernelArgs &a = *(const ConvKernelArgs *)(const ConvKernelArgs __attribute__((address_space(4))) *)address;
    const int block = __builtin_amdgcn_readfirstlane((int)blockIdx.x - first);
    if (block >= 8 * a.xcd_q + a.xcd_r) return;
    Body::template run<false>(a, reinterpret_cast<float *>(conv_smem), block, 0, 0);
}

}  // namespace ios
