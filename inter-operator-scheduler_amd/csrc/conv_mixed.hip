// Convolutions of different inputs and windows in a launch (conv_mixed_kernel), on the staged bodies.
#include "conv_window.h"
#include "conv_mixed.h"

namespace ios {

#define IOS_MIXED(...) {conv_mixed_kernel<ConvPipe<__VA_ARGS__, false, false>>, conv_mixed_kernel<ConvPipe<__VA_ARGS__, false, true>>},
#define IOS_PIPE3_MIXED(IDX, NAME, ...) IOS_MIXED(2, true, __VA_ARGS__)
#define IOS_PIPE_BF16_MIXED(IDX, NAME, ...) IOS_MIXED(1, false, __VA_ARGS__)
#define IOS_PIPE_FP16_MIXED(IDX, NAME, ...) IOS_MIXED(1, true, __VA_ARGS__)
extern const ConvMixedKernelFn kPipeMixedKernels[][2] = {IOS_PIPE3_VARIANTS(IOS_PIPE3_MIXED) IOS_PIPE_BF16_VARIANTS(IOS_PIPE_BF16_MIXED)
                                                          IOS_PIPE_FP16_VARIANTS(IOS_PIPE_FP16_MIXED)};

#define IOS_WINDOW3_MIXED(IDX, NAME, ...) conv_mixed_kernel<ConvWindow<2, true, __VA_ARGS__>>,
#define IOS_WINDOW_BF16_MIXED(IDX, NAME, ...) conv_mixed_kernel<ConvWindow<1, false, __VA_ARGS__>>,
#define IOS_WINDOW_FP16_MIXED(IDX, NAME, ...) conv_mixed_kernel<ConvWindow<1, true, __VA_ARGS__>>,
extern const ConvMixedKernelFn kWindowMixedKernels[] = {IOS_WINDOW3_VARIANTS(IOS_WINDOW3_MIXED) IOS_WINDOW_BF16_VARIANTS(IOS_WINDOW_BF16_MIXED)
                                                            IOS_WINDOW_FP16_VARIANTS(IOS_WINDOW_FP16_MIXED)};

}  // namespace ios
