// The kernels of conv_pipe.hip for inputs that need neither a ReLU nor channels masked.
#include "conv_pipe.h"
#include "conv_kernel.h"

namespace ios {

#define IOS_PIPE_KERNEL(TERMS, HALF, ...)                                                                                                       \
    {{conv_kernel<ConvPipe<TERMS, HALF, __VA_ARGS__, false, true>>, conv_kernel<ConvPipe<TERMS, HALF, __VA_ARGS__, false, true>, true>},             \
     {conv_kernel<ConvPipe<TERMS, HALF, __VA_ARGS__, true, true>>, conv_kernel<ConvPipe<TERMS, HALF, __VA_ARGS__, true, true>, true>}},
#define IOS_PIPE3_KERNEL(IDX, NAME, ...) IOS_PIPE_KERNEL(2, true, __VA_ARGS__)
#define IOS_PIPE_BF16_KERNEL(IDX, NAME, ...) IOS_PIPE_KERNEL(1, false, __VA_ARGS__)
#define IOS_PIPE_FP16_KERNEL(IDX, NAME, ...) IOS_PIPE_KERNEL(1, true, __VA_ARGS__)
extern const KernelPair kPipePlainKernels[][2] = {IOS_PIPE3_VARIANTS(IOS_PIPE3_KERNEL) IOS_PIPE_BF16_VARIANTS(IOS_PIPE_BF16_KERNEL)
                                                     IOS_PIPE_FP16_VARIANTS(IOS_PIPE_FP16_KERNEL)};

}  // namespace ios
