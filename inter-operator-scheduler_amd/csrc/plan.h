// Execution plan: the flat list of device operations, tensor views and the memory layout that a graph,
// block or stage document compiles to.  Planning is pure host code; nothing here touches the device.
//
// Memory model: one arena of 4-byte words.  Every operator output, temporary, filter, bias and split-K
// workspace is a region of it at a 256-byte aligned offset.  Tensors are NHWC, the channels of a pixel padded to a multiple of
// four (16-byte boundaries); a channel slice or a window of a concat buffer is again a view, so
//   * an identity with one input value is an alias (no memory, no work),
//   * a producer whose whole output is one term of a concat writes directly into the concat buffer,
//   * a channel slice of a merged convolution is read in place at any batch size,
//   * a ReLU that only feeds the next convolution of its Sequential is folded into that convolution's
//     input loader.
#pragma once

#include <functional>
#include <map>
#include <set>
#include <string>
#include <vector>

#include "json.h"
#include "kernels.h"

namespace ios {

constexpr int kMaxGroups = 16;   // concurrent groups (streams) per stage
constexpr int kMaxExtent = 1 << 16;     // image sides, filter sides, strides and padding a document may ask for
constexpr size_t kStagedBytes = size_t(256) << 20;   // largest transfer that is staged as a whole
constexpr size_t kDeliveredFloats = size_t(1) << 20;   // largest result that a pass writes to host memory by itself
constexpr int kMaxChannels = 1 << 20;   // channels of a tensor

// elements between the pixels of a tensor of its own
inline int padded_channels(int C) { return C < 3 ? C : (C + 3) & ~3; }

struct ViewRef {
    size_t base = 0;      // of the tensor the view lies in, in floats from the arena base
    int first = 0;        // channel of that tensor the view begins at
    int pstride = 0;      // elements between its pixels
    int C = 0, H = 0, W = 0;
    // The view's place in the tensor as if channels were the outermost dimension of an image: [offset, offset + C * H * W) and
    // bstride further for every image.  Two views of a tensor overlap where these ranges do (plans are described by them).
    size_t offset = 0;
    long long bstride = 0;
    ViewRef window(int begin, int end) const {
        ViewRef v = *this;
        v.offset += (size_t)begin * H * W;
        v.first += begin;
        v.C = end - begin;
        return v;
    }
    size_t image_floats() const { return (size_t)C * H * W; }
};

enum class OpKind { ConvMfma, ConvDepthwise, ConvDirect, Pool, GlobalPool, Nary, Unary };
const char *op_kind_name(OpKind kind);

struct PlanConv {
    std::string name;
    ConvProblem problem;
    size_t weight_off = 0, bias_off = 0;       // original layouts
    size_t packed_off = 0;                     // matrix path and depth-wise
    size_t ws_off = 0, ws_floats = 0;          // split-K only
    size_t ctr_off = 0, ctr_count = 0;         // split-K ticket counters (32-bit words at float offsets), zeroed at session setup
    ConvLaunch launch;
    bool matrix_path = false;
    // "average pool, then this convolution" run as "this convolution without bias and activation, then the pool, which adds
    // the bias and applies the activation": the convolution's launch reads OC zeros at zero_bias_off instead of the bias
    bool linear = false;
    size_t zero_bias_off = 0;
    bool thin = false;   // direct path: the kernel for 3 x 3 convolutions of 3-channel images (first layers at large batches)
};

struct PlanOp {
    OpKind kind;
    std::string node;     // operator name in the document
    int unit = -1;        // schedule unit (top-level operator) this op belongs to
    int stage = -1, group = -1;
    // position in the dependency order of the operations of its unit: operations of one unit on the same level are independent
    // of each other (the terms of a concatenation) and may run concurrently, a higher level reads what the lower ones wrote
    int level = 0;
    ViewRef in, out;
    int conv = -1;        // index into Plan::convs
    int bias_conv = -1;   // Pool behind a commuted convolution: out = act(pool(in) + bias of that convolution)
    PoolProblem pool{};
    std::vector<ViewRef> srcs;   // Nary: inputs; ConvDepthwise of a sum: the views it adds in its loader (else empty)
    int multiply = 0, accumulate = 0, act = 0;
    // ConvMfma of a residual unit: out = residual + act(conv + bias), then max(., 0) when post_relu
    bool has_residual = false;
    ViewRef residual;
    int post_relu = 0;
    // Where the operation reads and writes when the pass works on parts of the batch (operations of Plan::prefix_stages): a tensor
    // of the whole batch, or one that holds a part at a time.
    ViewRef part_in, part_out;
    bool part_in_whole = true, part_out_whole = true;
    int batch = -1;       // index into Plan::batches
    int moved_from = -1;  // its stage in the schedule, where a batch takes it ahead
    int scheduled_stage() const { return moved_from >= 0 ? moved_from : stage; }
    double flops = 0.0, bytes = 0.0;
};

// Convolutions that share a launch: of one view through the same window (launch_conv_batch), or mixed ones (launch_conv_mixed).  They run at
// the beginning of their stage, before its groups: an operation that the schedule puts into a later stage moves here.
struct PlanBatch {
    int stage = 0;
    int variant = -1;
    bool mixed = false;     // (a pool may be among its operations, the last of them)
    bool across_stages = false;   // the schedule puts some of them into later stages
    std::vector<int> ops;
};

struct Plan {
    int batch = 1;
    std::vector<PlanOp> ops;
    std::vector<PlanConv> convs;
    std::vector<std::vector<std::vector<int>>> stages;   // stage -> group -> op indices in launch order (without those of batches)
    std::vector<PlanBatch> batches;                      // by stage
    std::vector<std::string> unit_names;
    std::map<std::string, ViewRef> tensors;              // operator name -> materialised output view
    std::map<std::string, int> conv_index;               // convolution name -> index into convs
    ViewRef input, output;
    std::string input_name, output_name;
    size_t arena_floats = 0;
    // layout of the arena: [0, persistent_floats) filters, biases, packed filters and split-K ticket counters, which live as
    // long as the plan; behind them the regions of operator outputs, temporaries and split-K partial tiles.  With reuse
    // (planner option "arena_reuse"), regions whose lifetimes (first to last stage that touches them) do not intersect share
    // addresses; `overwritten` names the operators whose output does not survive to the end of a pass for that reason.
    size_t persistent_floats = 0;
    size_t activation_floats_without_reuse = 0;
    std::set<std::string> overwritten;
    bool output_single_group = true;                     // the last stage has one group
    // Leading stages of one group that may run on a part of the batch at a time, while the images behind it are still on their
    // way to the device (0: the input is too small for that, or the plan is not for a session that is given its input while it
    // works).  A tensor that only these stages read is then held for one part at a time: `in_parts` names the operators whose
    // output no pass on parts leaves as a whole.
    int prefix_stages = 0;
    std::vector<int> part_ends;   // images up to the end of each part
    size_t landing_off = 0;       // where the images of a plan with a prefix land, in the host's layout
    std::set<std::string> in_parts;
};

enum class PlanMode { Graph, Block, Stage };

// Resident: the input stays where it is for any number of passes.  InParts: the same, and it may arrive while the first stages work
// (Plan::prefix_stages).  Once: every pass is given its input, whose memory is free once its last reader has run.
enum class InputUse { Resident, InParts, Once };

// Picks the kernel configuration of a matrix-path convolution (closed-form model or measured).  `share` is the
// number of groups that run concurrently in the convolution's stage: a kernel that shares the device with
// share - 1 others should occupy about 1 / share of it rather than all of it.
typedef std::function<ConvLaunch(const ConvProblem &, int share)> LaunchChooser;

// Kernel configuration on which convolutions of one input (`mixed`: of any inputs and windows) run in a launch of their own, or -1 where
// they are faster by themselves; `share` of each as above, `stage`: in the schedule (those of one run beside each other where the share is
// more than one).  `remains`: other operations of their stage lose the launch that they shared with them.  `pool`: it runs beside mixed
// convolutions.
typedef std::function<int(const std::vector<ConvProblem> &, const std::vector<int> &share, const std::vector<int> &stage, bool remains, bool mixed,
                          const PoolProblem *pool)> BatchChooser;

// Compile a document.  `extra` is the input-shape document of stage mode ({name: [C, H, W]}).
// Throws std::runtime_error on malformed documents, unknown operator types, non-topological schedules
// and stages with too many groups.
// across_stages: convolutions of different stages may share a launch (as far as option batch_across_stages allows it).
Plan build_plan(PlanMode mode, const Json &doc, const Json *extra, int batch, const LaunchChooser &chooser, InputUse input = InputUse::Resident,
                const BatchChooser &batches = nullptr, bool across_stages = true);

std::string describe_plan(const Plan &plan);   // JSON array, one object per op

// Planner options that need no device: "arena_reuse" = "1" (default) | "0"; "thin_conv_min_pixels" = least number of output
// pixels (batch x OH x OW) from which a 3 x 3 convolution of a 3-channel image takes the output-bound direct kernel instead
// of the matrix path (default 2^18; a negative value disables it); "commute_pool_conv" = "1" (default) | "0": run "average
// pool that keeps the map size, then 1 x 1 convolution" as "convolution, then pool".  Returns false for an unknown key.
bool set_planner_option(const std::string &key, const std::string &value);
bool planner_arena_reuse();
long long planner_thin_conv_min_pixels();
int planner_host_split_k();   // option host_plan_split_k
bool planner_batch_convs();     // option batch_convs (default 1)
int planner_host_batches();     // option host_plan_batches
bool planner_commute_pool_conv();   // option commute_pool_conv (default 1): see PlanConv::linear

}  // namespace ios
