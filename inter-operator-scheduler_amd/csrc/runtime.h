// Device-side half of the runtime: the process-wide device context (stream pool, reusable arena, options,
// kernel-configuration cache) and Session, a plan bound to device memory that can be run, timed per
// stage and profiled per operation.
#pragma once

#include <hip/hip_runtime.h>

#include <map>
#include <memory>
#include <string>
#include <vector>

#include "plan.h"
#include "fused.h"
#include "host_io.h"

namespace ios {

void hip_check(hipError_t status, const char *what, const char *file, int line);
#define IOS_HIP(call) ::ios::hip_check((call), #call, __FILE__, __LINE__)

// Streams: one HIP stream per group, event fork/join.  Fused: one launch per level of a multi-group stage
// (see fused.h).  The *Graph modes capture the same issue sequence into a hipGraph and replay it.
enum class ExecMode { Streams, Graph, Fused, FusedGraph };

class DeviceContext {
public:
    static DeviceContext &get();   // initialises the device on first use

    int num_cus() const { return num_cus_; }
    const std::string &name() const { return name_; }
    const std::string &arch() const { return arch_; }
    hipStream_t stream(int group) { return streams_[group]; }
    HostStage &stage() { return stage_; }
    // the session whose last pass left its result in stage() (null: none)
    const void *result_owner = nullptr;
    // the sessions that laid out the shared arena and the static scratch last
    const void *shared_owner = nullptr, *static_owner = nullptr;
    int sessions = 0;   // that there are

    // a process-wide arena reused by the stateless latency / inference entry points
    float *shared_arena(size_t floats);
    void *shared_table(size_t bytes);   // companion buffer for the launch tables of such sessions

    void set_option(const std::string &key, const std::string &value);
    ExecMode exec_mode() const { return exec_mode_; }
    bool fused_executor() const { return exec_mode_ == ExecMode::Fused || exec_mode_ == ExecMode::FusedGraph; }
    bool autotune() const { return autotune_; }
    // split-K partial sums are added by a second kernel (Kernel), by the last block of a tile inside the convolution
    // kernel with the slices of a tile anywhere on the device (Inline), or the same with the slices of a tile numbered
    // onto one XCD, where they meet in that XCD's L2 (Xcd; the default when the placement probe at start-up found the
    // dispatcher's round-robin rule, and until a kernel reports a block somewhere else)
    enum class ReduceMode { Kernel, Inline, Xcd };
    ReduceMode reduce_mode() const { return reduce_mode_ == ReduceMode::Xcd && !xcd_usable_ ? ReduceMode::Inline : reduce_mode_; }
    bool inline_reduce() const { return reduce_mode_ != ReduceMode::Kernel; }
    // What the launchers take, for the mode in force and a launch on stream `group` of the pool.  The XCD a block lands
    // on depends on the stream (every stream starts its round-robin at an XCC of its own), so the XCD-local form needs
    // to know the stream; placement_known = false (kernels captured into a graph that forks: the replay runs them on
    // streams of its own) gives the device-wide form.
    SplitKReduce split_reduce(unsigned *counters, int group = 0, bool placement_known = true) const;
    // Throws when a kernel of the XCD-local form has reported a block on another XCC than the numbering assumes (results
    // of passes since the last check may be wrong); the form is switched off for the rest of the process first, so the
    // caller's next plan uses the device-wide form.
    void check_xcd_fault();
    bool xcd_usable() const { return xcd_usable_; }
    // testing aid: force one kernel configuration for every matrix-path convolution (-1 / 0 = off)
    int forced_variant() const { return forced_variant_; }
    int forced_split_k() const { return forced_split_k_; }
    std::string info_json() const;
    // changes with everything but the options that the choice of kernel configurations depends on
    std::string plan_token() const { return std::to_string(tuned.size()) + '/' + std::to_string(batched.size()) + (xcd_usable_ ? "x" : "-"); }

    // Kernel configuration for a matrix-path convolution: the measured best when autotuning is on (cached
    // per problem signature for the life of the process, and in the file named by IOS_TUNE_CACHE when set),
    // else the closed-form model; the testing overrides win over both.
    // `share` = number of groups running concurrently with this convolution (1 = alone on the device).
    // allow_tuning = false never measures (measuring allocates scratch tensors): a shape that has no cached winner
    // gets the closed-form choice.
    ConvLaunch choose_launch(const ConvProblem &p, int share, bool allow_tuning = true);

    // Kernel configuration on which these convolutions of one input share a launch, or -1 where the measurement finds them faster by
    // themselves (as choose_launch has them); see BatchChooser.  Without autotuning there are no batches, but on a forced configuration.
    int choose_batch(const std::vector<ConvProblem> &problems, const std::vector<int> &share, const std::vector<int> &stage, bool remains, bool mixed,
                     const PoolProblem *pool);

    // Static device scratch of the entry point that allocates nothing: address on device 0 (resolved once, when the
    // context is created) and size in bytes.
    float *static_scratch() const { return static_scratch_; }
    static size_t static_scratch_bytes();
    static constexpr int kShareClasses = 4;   // footprint budgets 1, 1/2, 1/4, 1/8 of the device
    struct TunedConv {
        ConvLaunch best[kShareClasses];
    };
    std::map<std::string, TunedConv> tuned;
    std::map<std::string, int> batched;   // choose_batch by its arguments

private:
    bool serves_batch(const std::vector<ConvProblem> &problems, int variant, bool mixed) const;
    int tune_batch(const std::vector<ConvProblem> &problems, const std::vector<int> &share, const std::vector<int> &stage, bool remains, bool mixed,
                   const PoolProblem *pool);
    DeviceContext();
    TunedConv tune_conv(const ConvProblem &p);
    float *tuning_buffer(int which, size_t floats);
    unsigned *tuning_counters(size_t count);
    float *static_scratch_ = nullptr;
    unsigned *tune_counters_ = nullptr;
    size_t tune_counter_count_ = 0;
    ReduceMode reduce_mode_ = ReduceMode::Xcd;
    bool xcd_usable_ = false;       // the start-up probe found blocks with equal index % 8 on one XCC, launch after launch
    unsigned xcd_map_[kMaxGroups] = {};   // per stream of the pool: that XCC per index % 8, four bits each
    unsigned *xcd_fault_ = nullptr; // one word of pinned host memory the kernels can write
    void probe_xcd_placement();
    int precision_ = PREC_FP32;   // operand type of the matrix-path convolutions (reduced-precision modes: PREC_BF16, PREC_FP16)
    bool share_cost_rule_ = true;   // share classes weigh time by the held share of the device (false: hard footprint budgets)
    int share_threads_per_cu_ = 1024;   // resident threads per compute unit the share-class budgets assume (four wavefronts per SIMD)
    void load_tune_cache();
    std::string settings_token() const;
    float *tune_buf_[4] = {nullptr, nullptr, nullptr, nullptr};
    size_t tune_floats_[4] = {0, 0, 0, 0};
    std::string tune_cache_path_;
    int num_cus_ = 0;
    std::string name_, arch_;
    hipStream_t streams_[kMaxGroups];
    HostStage stage_;
    float *arena_ = nullptr;
    size_t arena_floats_ = 0;
    void *table_ = nullptr;
    size_t table_bytes_ = 0;
    // defaults: fused stage launches (stream fork / join costs more than the batch-1 kernels it would overlap) and
    // measured kernel configurations, like the reference's exhaustive algorithm search on first sight of a shape
    ExecMode exec_mode_ = ExecMode::Fused;
    bool autotune_ = true;
    int forced_variant_ = -1;
    int forced_split_k_ = 0;
};

class Session {
public:
    // Where a session's device memory comes from: its own allocation, the context's shared arena (one such session at
    // a time), or the static scratch array (one at a time; such a session allocates nothing, creates no events, and
    // issues every operator on the main stream in schedule order whatever the executor option says).
    enum class Storage { Own, Shared, Static };
    // pack_filters: lay out whatever the filter regions hold, so that a pass without weights reads initialised memory; a
    // caller that sets the weights next packs with them (see finish_weights)
    Session(Plan plan, Storage storage, bool pack_filters = true);
    Session(Plan plan, bool shared) : Session(std::move(plan), shared ? Storage::Shared : Storage::Own) {}
    ~Session();
    void release() noexcept;   // frees device memory, events and the captured graph; safe to call twice
    Session(const Session &) = delete;
    Session &operator=(const Session &) = delete;

    const Plan &plan() const { return plan_; }

    void set_input(const float *host);
    // prints like the reference runtime, and skips the entry, when no convolution has a name
    void set_conv_weights(int count, char **names, float **weights, float **biases);
    void finish_weights();   // packs the filters of the convolutions that neither the constructor nor set_conv_weights has packed
    void get_output(float *host);
    // set_input, set_conv_weights, run and get_output in one, the pass following the weights as they arrive
    void infer(const float *input, int count, char **names, float **weights, float **biases, float *output);
    void get_tensor(const std::string &name, float *host);

    void run();   // one forward pass, synchronised
    void forward();       // one forward pass queued without waiting (stream launches or graph replay, by the execution mode)
    void synchronize();   // waits for everything queued
    // reference timing protocol for graphs / blocks: per repeat the mean of `number` individually
    // bracketed forward passes; optional per-stage times from events recorded after every stage
    void measure(int warmup, int number, int repeat, bool profile_stage, float *results, float *stage_results);
    // reference timing protocol for stage probes: `number` back-to-back passes in one bracket
    void measure_back_to_back(int warmup, int number, int repeat, float *results);
    void profile_ops(int warmup, int repeat, float *ms);
    // The kernel launches of one forward pass as the executor in force issues them (fused executors: one launch per
    // level of a multi-group stage, stand-alone kernels for single-group stages; stream executors: one per operation),
    // in issue order.
    struct LaunchRecord {
        int stage = 0;
        std::string kernel;      // e.g. "fused_kernel<512>", "conv_kernel<wq_m32n16_w8_t16>", "pool_kernel"
        std::vector<int> ops;    // indices into plan().ops
        int blocks = 0, threads = 0;
        int fused_level = -1;    // index into the stage's fused launches, -1 for a stand-alone kernel
        int batch = -1;          // index into plan().batches
    };
    std::vector<LaunchRecord> launches();
    std::string describe_launches();   // JSON array with the algorithmic flops and bytes of every launch
    // ms[i]: mean HIP-event time of launch i issued `repeat` times back to back on the launch stream
    void profile_launches(int warmup, int repeat, float *ms, int capacity);

private:
    void acquire(Storage storage, bool pack_filters);
    void setup(bool pack_filters);
    void pack(const PlanConv &conv, hipStream_t stream);
    void ensure_timers();
    void ensure_fork_events();
    // on stream `group` of the pool; images > 0: on that many images of the batch from `first` on
    void launch_op(const PlanOp &op, int group, int first = 0, int images = 0);
    TensorView part_of(const ViewRef &whole_view, const ViewRef &part_view, bool whole, int first, int images) const;
    void launch_batch(const PlanBatch &batch, int first = 0, int images = 0);   // on the main stream
    void launch_batches(size_t stage, int first = 0, int images = 0);           // those at the beginning of a stage
    void launch_scheduled_batches(size_t stage);
    unsigned *counters_of(const PlanConv &c) const;
    const float *bias_of(const PlanConv &c) const { return base_ + (c.linear ? c.zero_bias_off : c.bias_off); }
    void ready_executor();
    void enqueue(size_t first, bool stage_events);   // issue the stages from `first` on according to the execution mode
    void enqueue_stage(size_t s, bool timed = false);
    void enqueue_stage_streams(size_t s);
    void enqueue_stage_fused(size_t s);
    void enqueue_stage_serial(size_t s);
    void enqueue_prefix(size_t stages);
    size_t direct_stages() const;
    void build_fused();
    void build_graph(size_t first);
    void drop_graph() noexcept;
    void settle();
    void take_images(int first, int images, int chunk);
    void finish_pass();
    void advance();
    void attach();
    void copy_out(const ViewRef &view, float *host);
    TensorView tv(const ViewRef &v) const;

    Plan plan_;
    DeviceContext &ctx_;
    float *base_ = nullptr;
    bool owns_memory_ = false;
    bool static_ = false;
    bool released_ = false;
    std::vector<char> packed_;      // per convolution: its packed filters are laid out
    std::vector<int> arriving_;     // parts of the input on their way: images up to the end of each
    bool ran_in_parts_ = false;     // the last pass worked on parts of the batch as they arrived
    bool input_changed_ = false;    // the input or a weight has been set since the last pass
    bool advance_ = false;          // set_conv_weights issues the stages whose filters it has packed
    size_t next_stage_ = 0;
    unsigned delivered_pass_ = 0;   // the pass whose result is in the context's stage, where this session owns that
    bool fetches_result_ = true;    // the caller has fetched the last result (or there was none): the next pass delivers its own
    std::vector<hipEvent_t> fork_events_;                 // per stage (multi-group stages only)
    std::vector<std::vector<hipEvent_t>> join_events_;    // per stage, per extra group
    std::vector<hipEvent_t> stage_events_;                // per stage, profile mode
    hipEvent_t start_ = nullptr, stop_ = nullptr;
    struct FusedLaunch {
        int threads, first_item, num_items, total_blocks, smem_bytes;
        int single_op;   // >= 0: no fused launch, this plan operation is launched with its stand-alone kernel
        FusedHeader header;
        std::vector<int> ops;   // plan operations behind the items (a two-kernel split-K reduction names its convolution)
    };
    std::vector<std::vector<FusedLaunch>> fused_stages_;   // per stage; empty for stages whose operations all follow each other
    void *fused_items_ = nullptr;                          // device copy of all work items
    std::vector<WorkItem> fused_items_host_;
    bool fused_built_ = false;
    bool capturing_forks_ = false;   // a graph capture of the stream executor is under way (the replay chooses the streams)
    hipGraph_t graph_ = nullptr;
    ExecMode graph_mode_ = ExecMode::Graph;                // mode the captured graph was built for
    hipGraphExec_t graph_exec_ = nullptr;
};

}  // namespace ios
