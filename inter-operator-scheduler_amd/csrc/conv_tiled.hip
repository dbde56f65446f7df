// The LDS-tiled convolution kernels of conv_body.h, compiled apart from the others.
#include "conv_kernel.h"

namespace ios {

#define IOS_TILED_KERNEL(IDX, NAME, ...) {conv_kernel<ConvTiled<__VA_ARGS__>>, conv_kernel<ConvTiled<__VA_ARGS__>, true>},
extern const KernelPair kTiledKernels[] = {IOS_TILED_VARIANTS(IOS_TILED_KERNEL)};
#define IOS_SPLIT3_KERNEL(IDX, NAME, ...) {conv_kernel<ConvSplit3<__VA_ARGS__>>, conv_kernel<ConvSplit3<__VA_ARGS__>, true>},
extern const KernelPair kSplit3Kernels[] = {IOS_SPLIT3_VARIANTS(IOS_SPLIT3_KERNEL)};
#define IOS_SPLIT1_KERNEL(IDX, NAME, ...) {conv_kernel<ConvSplit3<__VA_ARGS__, 1>>, conv_kernel<ConvSplit3<__VA_ARGS__, 1>, true>},
extern const KernelPair kSplit1Kernels[] = {IOS_SPLIT1_VARIANTS(IOS_SPLIT1_KERNEL)};

}  // namespace ios
