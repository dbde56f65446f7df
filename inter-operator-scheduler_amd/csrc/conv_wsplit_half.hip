// Wave-split convolution kernels on the matrix instructions for half operands (conv_body.h), compiled apart from the others.
#include "conv_kernel.h"

namespace ios {

#define IOS_WSPLIT_X3S_KERNEL(IDX, NAME, TM, TN, NW, D) \
    {conv_kernel<ConvWsplit<16, TM, TN, NW, 8, true, D, 3>>, conv_kernel<ConvWsplit<16, TM, TN, NW, 8, true, D, 3>, true>},
extern const KernelPair kWsplitX3sKernels[] = {IOS_WSPLIT_X3S_VARIANTS(IOS_WSPLIT_X3S_KERNEL)};
#define IOS_WSPLIT_XH_KERNEL(IDX, NAME, TM, TN, NW, D) \
    {conv_kernel<ConvWsplit<32, TM, TN, NW, 8, true, D, 5>>, conv_kernel<ConvWsplit<32, TM, TN, NW, 8, true, D, 5>, true>},
extern const KernelPair kWsplitXhKernels[] = {IOS_WSPLIT_XH_VARIANTS(IOS_WSPLIT_XH_KERNEL)};

}  // namespace ios
