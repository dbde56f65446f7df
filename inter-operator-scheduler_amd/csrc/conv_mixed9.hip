// Convolutions of nine taps each, of different inputs, in a launch: windows that three rounds stage (conv_window9.hip).
#include "conv_window.h"
#include "conv_mixed.h"

namespace ios {

#define IOS_MIXED(TERMS, HALF, TMW, TNW, WM, WN, P_IT, NBUF) conv_mixed_kernel<ConvWindow<TERMS, HALF, TMW, TNW, WM, WN, short_rounds(P_IT), NBUF, 9>>,
#define IOS_WINDOW3_MIXED(IDX, NAME, ...) IOS_MIXED(2, true, __VA_ARGS__)
#define IOS_WINDOW_BF16_MIXED(IDX, NAME, ...) IOS_MIXED(1, false, __VA_ARGS__)
#define IOS_WINDOW_FP16_MIXED(IDX, NAME, ...) IOS_MIXED(1, true, __VA_ARGS__)
extern const ConvMixedKernelFn kWindow9MixedKernels[] = {IOS_WINDOW3_VARIANTS(IOS_WINDOW3_MIXED) IOS_WINDOW_BF16_VARIANTS(IOS_WINDOW_BF16_MIXED)
                                                             IOS_WINDOW_FP16_VARIANTS(IOS_WINDOW_FP16_MIXED)};

}  // namespace ios
