// Several convolutions of one input in a launch (conv_batch_kernel), on the staged bodies for 1 x 1 filters.
#include "conv_pipe.h"
#include "conv_kernel.h"

namespace ios {

#define IOS_BATCH(...) {conv_batch_kernel<ConvPipe<__VA_ARGS__, true, false>>, conv_batch_kernel<ConvPipe<__VA_ARGS__, true, true>>},
#define IOS_PIPE3_BATCH(IDX, NAME, ...) IOS_BATCH(2, true, __VA_ARGS__)
#define IOS_PIPE_BF16_BATCH(IDX, NAME, ...) IOS_BATCH(1, false, __VA_ARGS__)
#define IOS_PIPE_FP16_BATCH(IDX, NAME, ...) IOS_BATCH(1, true, __VA_ARGS__)
extern const ConvBatchKernelFn kPipeBatchKernels[][2] = {IOS_PIPE3_VARIANTS(IOS_PIPE3_BATCH) IOS_PIPE_BF16_VARIANTS(IOS_PIPE_BF16_BATCH)
                                                          IOS_PIPE_FP16_VARIANTS(IOS_PIPE_FP16_BATCH)};

}  // namespace ios
