// The convolution kernels that stage a window of the input (conv_window.h) for nine taps, compiled apart from the others.
#include "conv_window.h"
#include "conv_kernel.h"

namespace ios {

#define IOS_WINDOW_KERNEL(TERMS, HALF, ...) \
    {conv_kernel<ConvWindow<TERMS, HALF, __VA_ARGS__, 9>>, conv_kernel<ConvWindow<TERMS, HALF, __VA_ARGS__, 9>, true>},
#define IOS_WINDOW3_KERNEL(IDX, NAME, ...) IOS_WINDOW_KERNEL(2, true, __VA_ARGS__)
#define IOS_WINDOW_BF16_KERNEL(IDX, NAME, ...) IOS_WINDOW_KERNEL(1, false, __VA_ARGS__)
#define IOS_WINDOW_FP16_KERNEL(IDX, NAME, ...) IOS_WINDOW_KERNEL(1, true, __VA_ARGS__)
#define IOS_WINDOW3_SHORT(IDX, NAME, TMW, TNW, WM, WN, P_IT, NBUF) IOS_WINDOW_KERNEL(2, true, TMW, TNW, WM, WN, short_rounds(P_IT), NBUF)
#define IOS_WINDOW_BF16_SHORT(IDX, NAME, TMW, TNW, WM, WN, P_IT, NBUF) IOS_WINDOW_KERNEL(1, false, TMW, TNW, WM, WN, short_rounds(P_IT), NBUF)
#define IOS_WINDOW_FP16_SHORT(IDX, NAME, TMW, TNW, WM, WN, P_IT, NBUF) IOS_WINDOW_KERNEL(1, true, TMW, TNW, WM, WN, short_rounds(P_IT), NBUF)
extern const KernelPair kWindow9Kernels[] = {IOS_WINDOW3_VARIANTS(IOS_WINDOW3_KERNEL) IOS_WINDOW_BF16_VARIANTS(IOS_WINDOW_BF16_KERNEL)
                                                 IOS_WINDOW_FP16_VARIANTS(IOS_WINDOW_FP16_KERNEL)};
extern const KernelPair kWindow9ShortKernels[] = {IOS_WINDOW3_VARIANTS(IOS_WINDOW3_SHORT) IOS_WINDOW_BF16_VARIANTS(IOS_WINDOW_BF16_SHORT)
                                                      IOS_WINDOW_FP16_VARIANTS(IOS_WINDOW_FP16_SHORT)};

}  // namespace ios
