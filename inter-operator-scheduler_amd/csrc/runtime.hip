// Stage executor, timers and device context.
//
// A forward pass walks the plan's stages.  Fused executor (default): a multi-group stage is issued as one
// fused launch per chain position on the main stream (see build_fused).  Streams executor: group g of a stage
// is issued to stream g of a fixed pool; stream 0 is the main stream; a multi-group stage forks (the extra
// streams wait on an event recorded on the main stream) and joins (the main stream waits on one event per
// extra stream).  Either way stage boundaries are device-side dependencies and the host never blocks inside
// a pass.  The graph modes capture the same issue sequence once into a hipGraph and replay it.
//
// Timing follows the reference runtime (src/ios/ios_runtime.cu:1328-1455): graph / block latency is the
// mean over `number` individually bracketed passes per repeat, with optional per-stage times from events
// recorded on the main stream after every stage; stage probes time `number` back-to-back passes inside
// one event pair.
#include "runtime.h"

#include "fused.h"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <set>
#include <sstream>
#include <stdexcept>

namespace ios {

void hip_check(hipError_t status, const char *what, const char *file, int line) {
    if (status == hipSuccess) return;
    std::ostringstream os;
    os << "HIP failure " << hipGetErrorString(status) << " (" << (int)status << ") in " << what << " at " << file << ":" << line;
    throw std::runtime_error(os.str());
}

// ---- static scratch ----------------------------------------------------------------------------------------------
// Device memory of graph_inference_no_alloc: a session created with Storage::Static lays its whole arena (operator
// outputs, filters, packed filters, split-K partial tiles and ticket counters) out in this array instead of
// allocating.  The device holds it from the moment the library is loaded until the process ends.  In host code
// the array's name is only a handle for hipGetSymbolAddress; kernels and copies get the address resolved below.
constexpr size_t kStaticScratchBytes = size_t(256) << 20;
static __device__ __align__(256) float scratch[kStaticScratchBytes / sizeof(float)];

size_t DeviceContext::static_scratch_bytes() { return kStaticScratchBytes; }

// ---- device context --------------------------------------------------------------------------------------------
DeviceContext &DeviceContext::get() {
    static DeviceContext instance;
    return instance;
}

DeviceContext::DeviceContext() {
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count < 1) throw std::runtime_error("no HIP device available");
    IOS_HIP(hipSetDevice(0));
    hipDeviceProp_t prop;
    IOS_HIP(hipGetDeviceProperties(&prop, 0));
    num_cus_ = prop.multiProcessorCount;
    name_ = prop.name;
    arch_ = prop.gcnArchName;
    for (int i = 0; i < kMaxGroups; i++) IOS_HIP(hipStreamCreateWithFlags(&streams_[i], hipStreamNonBlocking));
    // the library runs on device 0 only, which is current here: its copy of the array is the one ever used
    IOS_HIP(hipGetSymbolAddress(reinterpret_cast<void **>(&static_scratch_), HIP_SYMBOL(scratch)));
    stage_.create();
    probe_xcd_placement();
    const char *mode = getenv("IOS_EXECUTOR");
    if (mode != nullptr) set_option("executor", mode);
    const char *tune = getenv("IOS_AUTOTUNE");
    if (tune != nullptr) set_option("autotune", tune);
    const char *cache = getenv("IOS_TUNE_CACHE");
    if (cache != nullptr && cache[0] != '\0') {
        tune_cache_path_ = cache;
        load_tune_cache();
    }
}

// ---- placement of workgroups on XCDs --------------------------------------------------------------------------------
// The XCD-local split-K relies on blocks with equal index % 8 running on one XCD (the dispatcher deals the workgroups of
// a launch round-robin).  The rule is checked here, on launches of several sizes, before anything uses it, and every block
// of such a launch checks its own XCC id again (xcd_enter).
__global__ void xcc_probe_kernel(unsigned *out) {
    if (threadIdx.x == 0) out[blockIdx.x] = xcc_id();
}

void DeviceContext::probe_xcd_placement() {
    xcd_usable_ = false;
    if (hipHostMalloc(reinterpret_cast<void **>(&xcd_fault_), 64, hipHostMallocMapped) != hipSuccess || xcd_fault_ == nullptr) {
        xcd_fault_ = nullptr;
        (void)hipGetLastError();
        return;
    }
    *xcd_fault_ = 0;
    constexpr int kMost = 1031;
    unsigned *device = nullptr;
    IOS_HIP(hipMalloc(reinterpret_cast<void **>(&device), kMost * sizeof(unsigned)));
    std::vector<unsigned> host(kMost);
    bool consistent = true;
    // Measured on MI355X: inside a launch, block b runs on XCC (first + b) % 8, and `first` is a constant of the stream
    // the launch goes to (launch after launch, alone or beside launches of other streams, also for the nodes that a
    // captured graph runs on the stream it is launched on).
    for (int g = 0; g < kMaxGroups; g++) {
        int seen[8] = {-1, -1, -1, -1, -1, -1, -1, -1};
        for (int blocks : {kMost, 8, 250}) {
            for (int threads : {64, 512}) {
                hipLaunchKernelGGL(xcc_probe_kernel, dim3(blocks), dim3(threads), 0, streams_[g], device);
                IOS_HIP(hipMemcpyAsync(host.data(), device, blocks * sizeof(unsigned), hipMemcpyDeviceToHost, streams_[g]));
                IOS_HIP(hipStreamSynchronize(streams_[g]));
                for (int b = 0; b < blocks; b++) {
                    if (seen[b & 7] < 0) seen[b & 7] = (int)host[b];
                    consistent = consistent && seen[b & 7] == (int)host[b] && host[b] < 16;
                }
            }
        }
        xcd_map_[g] = 0;
        for (int c = 0; c < 8; c++) xcd_map_[g] |= (unsigned)(seen[c] & 15) << (4 * c);
    }
    IOS_HIP(hipFree(device));
    xcd_usable_ = consistent;
}

SplitKReduce DeviceContext::split_reduce(unsigned *counters, int group, bool placement_known) const {
    SplitKReduce r;
    r.counters = inline_reduce() ? counters : nullptr;
    r.xcd_local = reduce_mode() == ReduceMode::Xcd && placement_known && group >= 0 && group < kMaxGroups;
    r.xcd_map = r.xcd_local ? xcd_map_[group] : 0;
    r.fault = xcd_fault_;
    return r;
}

void DeviceContext::check_xcd_fault() {
    if (xcd_fault_ == nullptr || *reinterpret_cast<volatile unsigned *>(xcd_fault_) == 0) return;
    *xcd_fault_ = 0;
    xcd_usable_ = false;
    tuned.clear();
    batched.clear();
    throw std::runtime_error("a split-K convolution found a workgroup on another XCD than the round-robin placement it relies on: results since the "
                             "last synchronisation may be wrong.  The XCD-local form is switched off for the rest of this process; create the session again");
}

// ---- kernel configuration choice ----------------------------------------------------------------------------------
static std::string conv_signature(const ConvProblem &p) {
    std::ostringstream os;
    os << p.B << ' ' << p.IC << ' ' << p.H << ' ' << p.W << ' ' << p.OC << ' ' << p.KH << ' ' << p.KW << ' ' << p.sh << ' ' << p.sw
       << ' ' << p.ph << ' ' << p.pw << ' ' << p.groups;
    return os.str();
}

// the measured winners of the share classes depend on these settings: they are part of every cache key
std::string DeviceContext::settings_token() const {
    std::ostringstream os;
    os << (share_cost_rule_ ? "cost" : "budget") << '/' << share_threads_per_cu_ << '/'
       << (reduce_mode() == ReduceMode::Xcd ? "xcd" : reduce_mode() == ReduceMode::Inline ? "inline" : "kernel")
       << (fused_executor() ? "" : "/own-launches");
    return os.str();
}

void DeviceContext::load_tune_cache() {
    FILE *f = fopen(tune_cache_path_.c_str(), "r");
    if (f == nullptr) return;
    // line: 12 problem integers, the settings token, then kShareClasses pairs (configuration name, split_k).  A line that
    // does not parse (truncated write, a configuration name this build no longer has) is skipped: its shape is measured again.
    char line[1024];
    while (fgets(line, sizeof(line), f) != nullptr) {
        // or "batch", the arguments of choose_batch and a configuration name or "none", with tabs between them
        if (strncmp(line, "batch\t", 6) == 0) {
            const std::string text(line + 6, strcspn(line + 6, "\n"));
            const size_t tab = text.find('\t');
            if (tab == std::string::npos) continue;
            const std::string name = text.substr(tab + 1);
            int variant = name == "none" ? -1 : -2;
            for (int i = 0; i < conv_num_variants(); i++)
                if (name == conv_variant(i).name && (conv_variant_batches(i) || conv_variant_mixes(i))) variant = i;
            if (variant >= -1) batched[text.substr(0, tab)] = variant;   // (whether it serves the shapes is seen when it is asked for)
            continue;
        }
        std::istringstream in(line);
        int v[12];
        bool ok = true;
        for (int i = 0; i < 12 && ok; i++) ok = static_cast<bool>(in >> v[i]);
        std::string token;
        ok = ok && static_cast<bool>(in >> token) && token.find('/') != std::string::npos;
        TunedConv entry;
        for (int c = 0; c < kShareClasses && ok; c++) {
            std::string name;
            int split = 0;
            ok = static_cast<bool>(in >> name >> split) && split >= 1 && split <= 64;
            int variant = -1;
            for (int i = 0; ok && i < conv_num_variants(); i++)
                if (name == conv_variant(i).name) variant = i;
            ok = ok && variant >= 0;
            entry.best[c].variant = variant;
            entry.best[c].split_k = split;
        }
        if (!ok) continue;
        for (int i : {0, 1, 2, 3, 4, 5, 6, 7, 8, 11}) ok = ok && v[i] >= 1;   // (the paddings may be 0)
        ok = ok && v[9] >= 0 && v[10] >= 0;
        if (!ok) continue;
        ConvProblem p{};
        p.B = v[0]; p.IC = v[1]; p.H = v[2]; p.W = v[3]; p.OC = v[4]; p.KH = v[5]; p.KW = v[6]; p.sh = v[7]; p.sw = v[8]; p.ph = v[9]; p.pw = v[10];
        p.groups = v[11];
        p.OH = (p.H + 2 * p.ph - p.KH) / p.sh + 1;
        p.OW = (p.W + 2 * p.pw - p.KW) / p.sw + 1;
        for (const ConvLaunch &l : entry.best) ok = ok && conv_variant_measured(p, l.variant) && conv_variant_takes(p, l.variant);
        if (!ok) continue;   // (a configuration that is not measured for this shape now: written by a build that had other kernels)
        std::ostringstream os;
        for (int i = 0; i < 12; i++) os << (i ? " " : "") << v[i];
        os << ' ' << token;
        // reduced-precision entries have their own keys
        if (conv_variant(entry.best[0].variant).precision == PREC_BF16) os << " bf16";
        if (conv_variant(entry.best[0].variant).precision == PREC_FP16) os << " fp16";
        tuned[os.str()] = entry;
    }
    fclose(f);
}

float *DeviceContext::tuning_buffer(int which, size_t floats) {
    if (floats > tune_floats_[which]) {
        IOS_HIP(hipDeviceSynchronize());
        if (tune_buf_[which] != nullptr) IOS_HIP(hipFree(tune_buf_[which]));
        tune_buf_[which] = nullptr;
        tune_floats_[which] = 0;
        const size_t want = floats + floats / 2 + 1024;
        IOS_HIP(hipMalloc(reinterpret_cast<void **>(&tune_buf_[which]), want * sizeof(float)));
        tune_floats_[which] = want;
        launch_fill_pattern(tune_buf_[which], want, 0x51f15e + which, streams_[0]);
        IOS_HIP(hipStreamSynchronize(streams_[0]));
    }
    return tune_buf_[which];
}

unsigned *DeviceContext::tuning_counters(size_t count) {
    if (count == 0) return nullptr;
    if (count > tune_counter_count_) {
        IOS_HIP(hipDeviceSynchronize());
        if (tune_counters_ != nullptr) IOS_HIP(hipFree(tune_counters_));
        tune_counters_ = nullptr;
        tune_counter_count_ = 0;
        const size_t want = count * 2 + 1024;
        IOS_HIP(hipMalloc(reinterpret_cast<void **>(&tune_counters_), want * sizeof(unsigned)));
        tune_counter_count_ = want;
        launch_fill_u32(tune_counters_, want, 0u, streams_[0]);
        IOS_HIP(hipStreamSynchronize(streams_[0]));
    }
    return tune_counters_;
}

DeviceContext::TunedConv DeviceContext::tune_conv(const ConvProblem &p) {
    // Like the reference's exhaustive algorithm search on first sight of a shape: run every kernel
    // configuration on scratch tensors of the real shape and keep the fastest.
    static const int kSplits[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32};
    const size_t kMaxWorkspace = size_t(96) << 20;   // floats
    TensorView x, y;
    x.C = p.IC; x.H = p.H; x.W = p.W; x.pstride = padded_channels(p.IC);
    y.C = p.OC; y.H = p.OH; y.W = p.OW; y.pstride = padded_channels(p.OC);
    x.ptr = tuning_buffer(0, (size_t)p.B * p.H * p.W * x.pstride + 64);   // (a 16-byte load may run past the last channel)
    y.ptr = tuning_buffer(1, (size_t)p.B * p.OH * p.OW * y.pstride);
    // Any values do for packed filters, except where two-term kernels read what belongs to a channel behind them: those are packed.
    const size_t packed_floats = conv_packed_floats_max(p);
    float *packed = tuning_buffer(2, 2 * packed_floats + p.OC + (size_t)p.OC * p.K());
    float *two_terms = packed + packed_floats, *bias = two_terms + packed_floats, *filters = bias + p.OC;
    int two_terms_cpad = 0;
    launch_fill_pattern(packed, 2 * packed_floats + p.OC + (size_t)p.OC * p.K(), 0x51f15e, streams_[0]);
    hipStream_t stream = streams_[0];
    struct EventPair {   // destroyed on every way out, a failing launch included
        hipEvent_t start = nullptr, stop = nullptr;
        ~EventPair() {
            if (start != nullptr) (void)hipEventDestroy(start);
            if (stop != nullptr) (void)hipEventDestroy(stop);
        }
    } events;
    IOS_HIP(hipEventCreate(&events.start));
    IOS_HIP(hipEventCreate(&events.stop));
    const hipEvent_t start = events.start, stop = events.stop;
    // one winner per footprint budget: the whole device, a half, a quarter, an eighth (threads in flight);
    // a convolution that shares its stage with other groups uses the winner of the matching budget
    const double capacity = (double)num_cus_ * (double)share_threads_per_cu_;
    struct Candidate {
        ConvLaunch launch;
        float ms;
        double footprint;
        bool fusable;
    };
    std::vector<Candidate> candidates;
    float fastest = 1e30f;
    constexpr float kQueuedMs = 0.008f, kLongMs = 0.04f;
    auto measure = [&](const ConvLaunch &l, int reps) {
        const size_t ws = conv_workspace_floats(p, l);
        float *workspace = ws ? tuning_buffer(3, ws) : nullptr;
        const SplitKReduce counters = split_reduce(tuning_counters(conv_counter_count(p, l)));
        const ConvVariant &cv = conv_variant(l.variant);
        if (cv.koct == 2 && cv.cpad != two_terms_cpad) {
            launch_pack_filters(p, l, filters, two_terms, stream);
            two_terms_cpad = cv.cpad;
        }
        auto issue = [&] { launch_conv_mfma(p, l, x, cv.koct == 2 ? two_terms : packed, filters, bias, y, workspace, counters, stream); };
        issue();   // warm-up
        // A launch costs the host 3 to 5 us, more than most kernels of a batch-1 network run: the device waits until all of
        // them are queued, so that the events time the kernels and not the host.  Where no kernel is that short, until the first.
        launch_delay(fastest < kQueuedMs || candidates.empty() ? reps + 3 : 2, stream);
        IOS_HIP(hipEventRecord(start, stream));
        for (int r = 0; r < reps; r++) issue();
        IOS_HIP(hipEventRecord(stop, stream));
        IOS_HIP(hipEventSynchronize(stop));
        float ms = 0.f;
        IOS_HIP(hipEventElapsedTime(&ms, start, stop));
        return ms / reps;
    };
    // first pass: every configuration and split factor, a few launches each
    for (int v = 0; v < conv_num_variants(); v++) {
        const ConvVariant &cv = conv_variant(v);
        if (cv.precision != precision_ || !conv_variant_measured(p, v) || !conv_variant_takes(p, v)) continue;   // the precision mode decides which family of configurations competes
        // tiles more than twice as tall / wide as the problem only waste lanes
        if (cv.BM >= 2 * p.OCg() + 32 || cv.BN >= 2 * p.Npix() + 32) continue;
        int last_effective = -1;
        for (int split : kSplits) {
            ConvLaunch l;
            l.variant = v;
            l.split_k = split;
            const int effective = conv_effective_split(p, l);
            if (effective == last_effective) continue;   // asks for more slices than there are K tiles
            last_effective = effective;
            if (conv_workspace_floats(p, l) > kMaxWorkspace) break;
            const float ms = measure(l, fastest < kQueuedMs ? 8 : fastest < kLongMs ? 4 : 2);
            const double footprint = (double)cv.threads() * ((p.OCg() + cv.BM - 1) / cv.BM) * (double)((p.Npix() + cv.BN - 1) / cv.BN) *
                                     p.groups * effective;
            candidates.push_back({l, ms, footprint, cv.fusable()});
            fastest = std::min(fastest, ms);
            if (ms > 3.f * fastest) break;   // more slices only add reduction work from here on
        }
    }
    // second pass: the fastest of every class again with more launches.  The first pass is noisy at 5-10 us, and many of the
    // configurations that are measured at all are close to each other.  Inception-v3 at batch 1, mean over 6 to 16 processes that
    // measure anew: 399 us with four launches in the first pass and three finalists, 396 with four and five, 392 with eight and five
    // (392 too with all 102 configurations, four launches and three finalists).
    constexpr int kFinalists = 5;
    std::sort(candidates.begin(), candidates.end(), [](const Candidate &a, const Candidate &b) { return a.ms < b.ms; });
    std::vector<char> refined(candidates.size(), 0);
    TunedConv result;
    bool found[kShareClasses];
    for (int c = 0; c < kShareClasses; c++) {
        // class 0 is unconstrained; the others accept kernels that fit their share of the device and, under the executors
        // that put the operators of a stage into one launch, can run inside a fused stage launch (the stream and graph
        // executors launch every operator by itself, so every configuration competes); a budget nobody fits takes the
        // fastest such configuration
        const bool any_kernel = !fused_executor();
        // A configuration of the wide-register fused family (three wavefronts per SIMD, items fetched from the table) only
        // competes when it runs for 9 us or more by itself: below that the family's slower start costs more than the
        // kernel gains.  (Inception-v3 at batch 1, two runs each: 423 and 413 us from 12 us on, 423 and 421 from 9; at batch 16 2015 and 2000 against
        // 1946 and 1953, ResNet-50 at batch 5 748 and 751 against 743 and 761.)
        constexpr float kWideMinMs = 0.009f;
        auto wide_too_short = [&](const Candidate &cand) {
            return !any_kernel && conv_variant(cand.launch.variant).needs_wide() && cand.ms < kWideMinMs;
        };
        auto eligible = [&](const Candidate &cand, bool fit) {
            if (c == 0) return true;
            if (wide_too_short(cand)) return false;
            return (cand.fusable || any_kernel) && (!fit || cand.footprint <= capacity / (1 << c));
        };
        found[c] = false;
        if (c > 0 && share_cost_rule_) {
            // soft form: time weighted by the share of the device the kernel holds while 2^c - 1 neighbours want theirs
            auto score = [&](const Candidate &cand) { return cand.ms * (1.0 + ((1 << c) - 1) * cand.footprint / capacity); };
            std::vector<size_t> order;
            for (size_t i = 0; i < candidates.size(); i++)
                if ((candidates[i].fusable || any_kernel) && !wide_too_short(candidates[i])) order.push_back(i);
            std::sort(order.begin(), order.end(), [&](size_t a, size_t b) { return score(candidates[a]) < score(candidates[b]); });
            double best = 1e300;
            for (size_t n = 0; n < order.size() && n < kFinalists; n++) {
                Candidate &cand = candidates[order[n]];
                if (!refined[order[n]]) {
                    cand.ms = std::min(cand.ms, measure(cand.launch, 16));
                    refined[order[n]] = 1;
                }
                if (score(cand) < best) {
                    best = score(cand);
                    result.best[c] = cand.launch;
                    found[c] = true;
                }
            }
        }
        for (int pass = 0; pass < 2 && !found[c]; pass++) {
            int taken = 0;
            float best = 1e30f;
            for (size_t i = 0; i < candidates.size() && taken < kFinalists; i++) {
                if (!eligible(candidates[i], pass == 0)) continue;
                taken++;
                if (!refined[i]) {
                    candidates[i].ms = std::min(candidates[i].ms, measure(candidates[i].launch, 16));
                    refined[i] = 1;
                }
                if (candidates[i].ms < best) {
                    best = candidates[i].ms;
                    result.best[c] = candidates[i].launch;
                    found[c] = true;
                }
            }
        }
        if (!found[c]) result.best[c] = conv_pick_launch(p, std::max(1, num_cus_ >> c), c > 0, precision_);
    }
    // A convolution large enough for a kernel that no fused launch can hold is launched by itself also where it shares its stage:
    // when that kernel and the gap in front of it take less than the device time of the best fusable one, which is its time
    // or, where its blocks do not fill the device, their share of it.  (Allowing 5 us for the gap; Inception-v3 under the greedy
    // schedule: bfloat16 at batch 24 1970 -> 1840 us, fp32 at batch 32 3335 -> 3270, half at batch 12 1115 -> 1090; SqueezeNet, half,
    // batch 50 585 -> 480.  With 3 us the middle sizes lose up to 1 %, with 8 the small maps 7 %.)
    constexpr float kGapMs = 0.005f;
    if (fused_executor() && found[0] && !conv_variant(result.best[0].variant).fusable()) {
        auto device_time = [&](const ConvLaunch &l) {
            for (const Candidate &cand : candidates)
                if (cand.launch.variant == l.variant && cand.launch.split_k == l.split_k) return cand.ms * (float)std::min(1.0, cand.footprint / capacity);
            return 0.f;
        };
        float alone = 0.f;
        for (const Candidate &cand : candidates)
            if (cand.launch.variant == result.best[0].variant && cand.launch.split_k == result.best[0].split_k) alone = cand.ms;
        for (int c = 1; c < kShareClasses; c++)
            if (found[c] && alone + kGapMs < device_time(result.best[c])) result.best[c] = result.best[0];
    }
    if (!tune_cache_path_.empty()) {
        FILE *f = fopen(tune_cache_path_.c_str(), "a");
        if (f != nullptr) {
            fprintf(f, "%s %s", conv_signature(p).c_str(), settings_token().c_str());
            for (int c = 0; c < kShareClasses; c++) fprintf(f, " %s %d", conv_variant(result.best[c].variant).name, result.best[c].split_k);
            fprintf(f, "\n");
            fclose(f);
        }
    }
    return result;
}

ConvLaunch DeviceContext::choose_launch(const ConvProblem &p, int share, bool allow_tuning) {
    int cls = 0;
    while (cls + 1 < kShareClasses && (1 << (cls + 1)) <= share) cls++;   // floor(log2(share)), capped
    ConvLaunch launch;
    bool chosen = false;
    if (autotune_) {
        const std::string key = conv_signature(p) + " " + settings_token() + (precision_ == PREC_BF16 ? " bf16" : precision_ == PREC_FP16 ? " fp16" : "");
        auto it = tuned.find(key);
        if (it == tuned.end() && allow_tuning) it = tuned.emplace(key, tune_conv(p)).first;
        if (it != tuned.end()) {
            launch = it->second.best[cls];
            chosen = true;
        }
    }
    if (!chosen) {
        launch = conv_pick_launch(p, std::max(1, num_cus_ >> cls), cls > 0, precision_);
    }
    if (forced_variant_ >= 0) launch.variant = forced_variant_;
    if (forced_split_k_ > 0) launch.split_k = forced_split_k_;
    return launch;
}

static WorkItem conv_work_item(const ConvDispatch &d) {
    WorkItem item;
    memset(&item, 0, sizeof(WorkItem));
    item.kind = WORK_CONV;
    item.variant = d.variant;
    item.threads = d.threads;
    item.tiles = d.tiles;
    item.groups = d.groups;
    item.div_tiles = make_fast_div((unsigned)d.tiles);
    item.div_groups = make_fast_div((unsigned)d.groups);
    item.num_blocks = d.grid_blocks();
    item.conv = d.args;
    return item;
}

// a configuration that a launch of these convolutions may be measured on
bool DeviceContext::serves_batch(const std::vector<ConvProblem> &problems, int variant, bool mixed) const {
    if (conv_variant(variant).precision != precision_ || !(mixed ? conv_variant_mixes(variant) : conv_variant_batches(variant))) return false;
    for (const ConvProblem &p : problems)
        if (!(mixed ? conv_mixable(p, variant) : conv_variant_precise(p, variant))) return false;
    return true;
}

// Both ways on scratch tensors of the real shapes: every convolution as it runs without a batch (those of one stage whose share is more than
// one beside each other, in a fused launch or on streams, as the executor has them), and all of them in a launch on every configuration that
// has such a kernel.
int DeviceContext::tune_batch(const std::vector<ConvProblem> &problems, const std::vector<int> &share, const std::vector<int> &stage, bool remains, bool mixed,
                              const PoolProblem *pool) {
    const size_t count = problems.size();
    bool parallel = false;
    for (int s : share) parallel = parallel || s > 1;
    if (mixed && parallel && !fused_executor()) return -1;   // (they run beside each other, on streams)
    std::vector<ConvLaunch> alone;
    for (size_t i = 0; i < count; i++) alone.push_back(choose_launch(problems[i], share[i]));
    std::vector<TensorView> x(count), y(count);
    std::vector<size_t> x_at(count);
    size_t x_floats = 0;
    for (size_t i = 0; i < count; i++) {
        const ConvProblem &p = problems[i];
        x[i].C = p.IC; x[i].H = p.H; x[i].W = p.W; x[i].pstride = padded_channels(p.IC);
        if (!mixed && i > 0) continue;   // (one input)
        x_at[i] = x_floats;
        x_floats += ((size_t)p.B * p.H * p.W * x[i].pstride + 64 + 63) & ~size_t(63);
    }
    MixedPool beside{};
    size_t pool_x_at = 0, pool_y_at = 0;
    if (pool != nullptr) {
        beside.p = *pool;
        beside.x.C = beside.y.C = pool->C;
        beside.x.H = pool->H; beside.x.W = pool->W; beside.y.H = pool->OH; beside.y.W = pool->OW;
        beside.x.pstride = beside.y.pstride = padded_channels(pool->C);
        pool_x_at = x_floats;
        x_floats += ((size_t)pool->B * pool->H * pool->W * beside.x.pstride + 64 + 63) & ~size_t(63);
        pool_y_at = x_floats;
        x_floats += ((size_t)pool->B * pool->OH * pool->OW * beside.y.pstride + 64 + 63) & ~size_t(63);
    }
    float *x_memory = tuning_buffer(0, x_floats);
    beside.x.ptr = x_memory + pool_x_at;
    beside.y.ptr = x_memory + pool_y_at;
    for (size_t i = 0; i < count; i++) x[i].ptr = x_memory + x_at[i];
    std::vector<size_t> y_at(count), packed_at(count), filters_at(count), ws_at(count), ctr_at(count);
    size_t y_floats = 0, floats = 0, ws_floats = 0, counters = 0, items_at = 0;
    for (size_t i = 0; i < count; i++) {
        const ConvProblem &q = problems[i];
        y[i].C = q.OC; y[i].H = q.OH; y[i].W = q.OW; y[i].pstride = padded_channels(q.OC);
        y_at[i] = y_floats;
        y_floats += ((size_t)q.B * q.OH * q.OW * y[i].pstride + 63) & ~size_t(63);
        packed_at[i] = floats;
        floats += (conv_packed_floats_max(q) + 63) & ~size_t(63);
        filters_at[i] = floats;   // (the first of them serve as its bias)
        floats += ((size_t)q.OC * q.K() + 63) & ~size_t(63);
        ws_at[i] = ws_floats;
        ws_floats += conv_workspace_floats(q, alone[i]);
        ctr_at[i] = counters;
        counters += conv_counter_count(q, alone[i]);
    }
    items_at = floats;
    floats += ((count + 1) * sizeof(WorkItem) + sizeof(float) - 1) / sizeof(float);
    float *y_memory = tuning_buffer(1, y_floats), *memory = tuning_buffer(2, floats), *workspace = ws_floats ? tuning_buffer(3, ws_floats) : nullptr;
    unsigned *tickets = tuning_counters(counters);
    hipStream_t stream = streams_[0];
    launch_fill_pattern(memory, items_at, 0x51f15e, stream, 0.5f);
    for (size_t i = 0; i < count; i++) y[i].ptr = y_memory + y_at[i];
    struct EventPair {   // destroyed on every way out, a failing launch included
        hipEvent_t start = nullptr, stop = nullptr;
        ~EventPair() {
            if (start != nullptr) (void)hipEventDestroy(start);
            if (stop != nullptr) (void)hipEventDestroy(stop);
        }
    } events;
    IOS_HIP(hipEventCreate(&events.start));
    IOS_HIP(hipEventCreate(&events.stop));
    auto measure = [&](int reps, int launches, const std::function<void()> &issue) {
        issue();
        launch_delay(reps * launches + 3, stream);   // (as in tune_conv: the events time the kernels and not the host)
        IOS_HIP(hipEventRecord(events.start, stream));
        for (int r = 0; r < reps; r++) issue();
        IOS_HIP(hipEventRecord(events.stop, stream));
        IOS_HIP(hipEventSynchronize(events.stop));
        float ms = 0.f;
        IOS_HIP(hipEventElapsedTime(&ms, events.start, events.stop));
        return ms / reps;
    };
    constexpr int kReps = 8;
    // by themselves
    struct Level {   // what a stage has in a fused launch
        std::vector<WorkItem> items;
        std::vector<size_t> members;
        FusedHeader header{};
        int blocks = 0, smem_bytes = 0, threads = 256;
        bool wide = false, pool = false;
        size_t first_item = 0;
        void add(WorkItem item) {
            item.first_block = blocks;
            header.first_block[items.size()] = blocks;
            blocks += item.num_blocks;
            items.push_back(item);
            header.num_items = (int)items.size();
        }
    };
    std::map<int, Level> levels;
    std::vector<size_t> single;
    for (size_t i = 0; i < count; i++) {
        launch_pack_filters(problems[i], alone[i], memory + filters_at[i], memory + packed_at[i], stream);
        const ConvDispatch d = make_conv_dispatch(problems[i], alone[i], x[i], memory + packed_at[i], memory + filters_at[i], memory + filters_at[i], y[i],
                                                  workspace != nullptr ? workspace + ws_at[i] : nullptr, split_reduce(tickets != nullptr ? tickets + ctr_at[i] : nullptr));
        if (share[i] <= 1 || !fused_executor() || !conv_variant(d.variant).fusable() || d.has_reduce) {
            single.push_back(i);
            continue;
        }
        Level &level = levels[stage[i]];
        level.add(conv_work_item(d));
        level.members.push_back(i);
        level.smem_bytes = std::max(level.smem_bytes, d.smem_bytes);
        level.threads = std::max(level.threads, d.threads);
        level.wide = level.wide || conv_variant(d.variant).needs_wide();
    }
    for (auto it = levels.begin(); it != levels.end();) {   // (no fused launch holds both: build_fused launches such a level one by one)
        const Level &level = it->second;
        if (level.wide && level.threads > 512) {
            single.insert(single.end(), level.members.begin(), level.members.end());
            it = levels.erase(it);
        } else {
            ++it;
        }
    }
    const bool pool_alone = pool != nullptr && levels.empty();
    if (pool != nullptr && !pool_alone) {   // (of the stage that all members are of)
        Level &level = levels.begin()->second;
        WorkItem item;
        memset(&item, 0, sizeof(item));
        item.kind = WORK_POOL;
        item.pool = make_pool_args(beside.p, beside.x, beside.y, false, &item.num_blocks);
        item.num_blocks = std::max(1, (item.num_blocks * 256 + level.threads - 1) / level.threads);
        item.threads = level.threads;
        level.add(item);
    }
    std::vector<WorkItem> items;
    for (auto &entry : levels) {
        entry.second.first_item = items.size();
        items.insert(items.end(), entry.second.items.begin(), entry.second.items.end());
    }
    WorkItem *device_items = reinterpret_cast<WorkItem *>(memory + items_at);
    if (!items.empty()) stage_.upload(device_items, items.data(), items.size() * sizeof(WorkItem), stream);
    struct Joins {   // of streams beside the main one
        std::vector<hipEvent_t> events;
        ~Joins() {
            for (hipEvent_t event : events) (void)hipEventDestroy(event);
        }
    } joins;
    auto beside_others = [&](size_t i) {   // on a stream of its own
        return !fused_executor() && share[i] > 1 && std::count(stage.begin(), stage.end(), stage[i]) > 1;
    };
    for (size_t i = 0; i <= count; i++) {   // (one event to fork)
        joins.events.push_back(nullptr);
        IOS_HIP(hipEventCreateWithFlags(&joins.events.back(), hipEventDisableTiming));
    }
    const bool placement_known = !(parallel && exec_mode_ == ExecMode::Graph);   // (captured forks run on streams that nobody knows)
    auto launch_alone = [&](size_t i, size_t group) {
        launch_conv_mfma(problems[i], alone[i], x[i], memory + packed_at[i], memory + filters_at[i], memory + filters_at[i], y[i],
                         workspace != nullptr ? workspace + ws_at[i] : nullptr,
                         split_reduce(tickets != nullptr ? tickets + ctr_at[i] : nullptr, (int)group, placement_known), streams_[group]);
    };
    const int launches_apart = (int)(3 * single.size() + levels.size() + 2);   // (the joins among them)
    const float apart = measure(kReps, launches_apart, [&] {
        if (pool_alone) launch_pool(beside.p, beside.x, beside.y, stream);
        for (const auto &entry : levels) {
            const Level &level = entry.second;
            launch_fused(level.threads, device_items + level.first_item, items.data() + level.first_item, level.header, level.blocks, level.smem_bytes, num_cus_, stream);
        }
        for (size_t n = 0; n < single.size(); n++) {
            const size_t i = single[n];
            if (!beside_others(i)) {
                launch_alone(i, 0);
                continue;
            }
            size_t end = n;   // (members come by stage)
            while (end < single.size() && stage[single[end]] == stage[i] && beside_others(single[end])) end++;
            IOS_HIP(hipEventRecord(joins.events[count], stream));
            for (size_t m = n + 1; m < end; m++) IOS_HIP(hipStreamWaitEvent(streams_[m - n], joins.events[count], 0));
            for (size_t m = n; m < end; m++) launch_alone(single[m], m - n);
            for (size_t m = n + 1; m < end; m++) {
                IOS_HIP(hipEventRecord(joins.events[m], streams_[m - n]));
                IOS_HIP(hipStreamWaitEvent(stream, joins.events[m], 0));
            }
            n = end - 1;
        }
    });
    // together
    float best = 1e30f;
    int variant = -1;
    std::vector<ConvBatchMember> members(count);
    for (size_t i = 0; i < count; i++) members[i] = {problems[i], memory + packed_at[i], memory + filters_at[i], memory + filters_at[i], x[i], y[i]};
    bool packed = false;
    for (int v = 0; v < conv_num_variants(); v++) {
        if (!serves_batch(problems, v, mixed)) continue;
        ConvLaunch l;
        l.variant = v;
        for (size_t i = 0; i < count && !packed; i++) launch_pack_filters(problems[i], l, memory + filters_at[i], memory + packed_at[i], stream);
        packed = true;   // (they all read the same layout)
        const float ms = measure(kReps, 1, [&] {
            if (mixed) launch_conv_mixed(members.data(), (int)count, pool != nullptr ? &beside : nullptr, v, stream);
            else launch_conv_batch(members.data(), (int)count, v, stream);
        });
        if (ms < best) {
            best = ms;
            variant = v;
        }
    }
    // What is left of a stage takes a launch of its own: 3 us.  A gain within the noise of the measurement is none.
    constexpr float kLaunchMs = 0.003f, kNoise = 0.97f;
    return best + (remains ? kLaunchMs : 0.f) < kNoise * apart ? variant : -1;
}

int DeviceContext::choose_batch(const std::vector<ConvProblem> &problems, const std::vector<int> &share, const std::vector<int> &stage, bool remains, bool mixed,
                                const PoolProblem *pool) {
    if (forced_variant_ >= 0) {
        const bool serves = mixed ? serves_batch(problems, forced_variant_, true) : conv_variant_batches(forced_variant_);
        return forced_split_k_ <= 1 && serves ? forced_variant_ : -1;
    }
    if (!autotune_ || forced_split_k_ > 0) return -1;
    std::string key = (mixed ? "mixed " : "") + settings_token() + (precision_ == PREC_BF16 ? " bf16" : precision_ == PREC_FP16 ? " fp16" : "") + (remains ? " remains" : "");
    const std::set<int> stages(stage.begin(), stage.end());
    bool parallel = false;
    for (int s : share) parallel = parallel || s > 1;
    for (size_t i = 0; i < problems.size(); i++) {
        key += " | " + conv_signature(problems[i]) + " " + std::to_string(share[i]);
        if (parallel) key += "@" + std::to_string(std::distance(stages.begin(), stages.find(stage[i])));   // (who runs beside whom)
    }
    if (pool != nullptr) {
        key += " | pool";
        for (int n : {pool->C, pool->H, pool->W, pool->KH, pool->KW, pool->sh, pool->sw, pool->ph, pool->pw, pool->is_max})
            key += ' ' + std::to_string(n);
    }
    auto it = batched.find(key);
    if (it != batched.end() && it->second >= 0) {   // (a saved choice that would not be measured here: written by a build that had other kernels)
        if (!serves_batch(problems, it->second, mixed)) {
            batched.erase(it);
            it = batched.end();
        }
    }
    if (it == batched.end()) {
        it = batched.emplace(key, tune_batch(problems, share, stage, remains, mixed, pool)).first;
        FILE *f = tune_cache_path_.empty() ? nullptr : fopen(tune_cache_path_.c_str(), "a");
        if (f != nullptr) {
            fprintf(f, "batch\t%s\t%s\n", key.c_str(), it->second >= 0 ? conv_variant(it->second).name : "none");
            fclose(f);
        }
    }
    return it->second;
}

float *DeviceContext::shared_arena(size_t floats) {
    if (floats > arena_floats_) {
        IOS_HIP(hipDeviceSynchronize());
        if (arena_ != nullptr) IOS_HIP(hipFree(arena_));
        arena_ = nullptr;
        arena_floats_ = 0;
        const size_t want = floats + floats / 4 + (1u << 20);
        IOS_HIP(hipMalloc(reinterpret_cast<void **>(&arena_), want * sizeof(float)));
        arena_floats_ = want;
        // latency probes run on whatever the arena holds; start from finite, varied values
        launch_fill_pattern(arena_, arena_floats_, 0x1234567u, streams_[0]);
        IOS_HIP(hipStreamSynchronize(streams_[0]));
    }
    return arena_;
}

void *DeviceContext::shared_table(size_t bytes) {
    if (bytes > table_bytes_) {
        IOS_HIP(hipDeviceSynchronize());
        if (table_ != nullptr) IOS_HIP(hipFree(table_));
        table_ = nullptr;
        table_bytes_ = 0;
        const size_t want = bytes * 2 + 4096;
        IOS_HIP(hipMalloc(&table_, want));
        table_bytes_ = want;
    }
    return table_;
}

void DeviceContext::set_option(const std::string &key, const std::string &value) {
    if (key == "executor") {
        if (value == "streams") exec_mode_ = ExecMode::Streams;
        else if (value == "graph") exec_mode_ = ExecMode::Graph;
        else if (value == "fused") exec_mode_ = ExecMode::Fused;
        else if (value == "fused_graph") exec_mode_ = ExecMode::FusedGraph;
        else throw std::runtime_error("option executor: expected streams, graph, fused or fused_graph, got '" + value + "'");
    } else if (key == "autotune") {
        autotune_ = !(value == "0" || value == "false" || value == "off" || value.empty());
    } else if (key == "conv_variant") {
        const int v = atoi(value.c_str());
        if (v < -1 || v >= conv_num_variants()) throw std::runtime_error("option conv_variant: index out of range");
        forced_variant_ = v;
    } else if (key == "conv_split_k") {
        const int v = atoi(value.c_str());
        if (v < 0 || v > 64) throw std::runtime_error("option conv_split_k: expected 0..64");
        forced_split_k_ = v;
    } else if (key == "share_rule") {
        if (value == "cost") share_cost_rule_ = true;
        else if (value == "budget") share_cost_rule_ = false;
        else throw std::runtime_error("option share_rule: expected cost or budget");
    } else if (key == "share_threads_per_cu") {
        const int v = atoi(value.c_str());
        if (v < 64 || v > 4096) throw std::runtime_error("option share_threads_per_cu: expected 64..4096");
        share_threads_per_cu_ = v;
    } else if (key == "precision") {
        if (value == "fp32") precision_ = PREC_FP32;
        else if (value == "bf16") precision_ = PREC_BF16;
        else if (value == "fp16") precision_ = PREC_FP16;
        else throw std::runtime_error("option precision: expected fp32, bf16 or fp16, got '" + value + "'");
    } else if (key == "split_k_reduce") {
        if (value == "xcd") reduce_mode_ = ReduceMode::Xcd;   // (falls back to inline where the placement probe failed)
        else if (value == "inline") reduce_mode_ = ReduceMode::Inline;
        else if (value == "kernel") reduce_mode_ = ReduceMode::Kernel;
        else throw std::runtime_error("option split_k_reduce: expected xcd, inline or kernel, got '" + value + "'");
    } else if (key == "host_threads") {
        const int v = atoi(value.c_str());
        if (v < 0 || v > 1024) throw std::runtime_error("option host_threads: expected 0..1024");
        HostCopier::get().set_threads(v);
    } else if (key == "release_staging") {
        IOS_HIP(hipDeviceSynchronize());
        stage_.give_back();
    } else if (key == "clear_tuning") {
        tuned.clear();
        batched.clear();
    } else {
        throw std::runtime_error("unknown option '" + key + "'");
    }
}

std::string DeviceContext::info_json() const {
    std::ostringstream os;
    os << "{\"name\":\"" << name_ << "\",\"arch\":\"" << arch_ << "\",\"compute_units\":" << num_cus_
       << ",\"executor\":\"" << (exec_mode_ == ExecMode::Graph ? "graph" : exec_mode_ == ExecMode::Fused ? "fused" : exec_mode_ == ExecMode::FusedGraph ? "fused_graph" : "streams") << "\",\"autotune\":" << (autotune_ ? "true" : "false")
       << ",\"split_k_reduce\":\"" << (reduce_mode_ == ReduceMode::Xcd ? "xcd" : reduce_mode_ == ReduceMode::Inline ? "inline" : "kernel") << "\""
       << ",\"xcd_placement_probe\":" << (xcd_usable_ ? "true" : "false") << ",\"xcd_map\":" << xcd_map_[0]
       << ",\"precision\":\"" << (precision_ == PREC_BF16 ? "bf16" : precision_ == PREC_FP16 ? "fp16" : "fp32") << "\""
       << ",\"conv_variant\":" << forced_variant_ << ",\"conv_split_k\":" << forced_split_k_
       << ",\"staged_bytes\":" << stage_.staged_bytes() << ",\"host_threads\":" << HostCopier::get().threads()
       << ",\"arena_reuse\":" << (planner_arena_reuse() ? "true" : "false")
       << ",\"max_groups\":" << kMaxGroups << ",\"conv_variants\":[";
    for (int i = 0; i < conv_num_variants(); i++) os << (i ? "," : "") << '"' << conv_variant(i).name << '"';
    os << "]}";
    return os.str();
}

// ---- session ---------------------------------------------------------------------------------------------------------
Session::Session(Plan plan, Storage storage, bool pack_filters) : plan_(std::move(plan)), ctx_(DeviceContext::get()) {
    ctx_.sessions++;
    try {
        acquire(storage, pack_filters);
    } catch (...) {
        release();   // the destructor does not run for a constructor that throws
        throw;
    }
}

void Session::acquire(Storage storage, bool pack_filters) {
    if (storage == Storage::Static) {
        const size_t need = plan_.arena_floats * sizeof(float);
        if (need > DeviceContext::static_scratch_bytes())
            throw std::runtime_error("graph needs " + std::to_string(need) + " bytes of device memory at this batch size; the static scratch of "
                                     "graph_inference_no_alloc holds " + std::to_string(DeviceContext::static_scratch_bytes()));
        base_ = ctx_.static_scratch();
        static_ = true;
        ctx_.static_owner = this;
    } else if (storage == Storage::Shared) {
        base_ = ctx_.shared_arena(plan_.arena_floats);
        ctx_.shared_owner = this;
    } else {
        IOS_HIP(hipMalloc(reinterpret_cast<void **>(&base_), std::max<size_t>(plan_.arena_floats, 64) * sizeof(float)));
        owns_memory_ = true;
    }
    setup(pack_filters);
}

Session::~Session() { release(); }

void Session::release() noexcept {
    if (ctx_.result_owner == this) ctx_.result_owner = nullptr;
    (void)hipDeviceSynchronize();
    drop_graph();
    if (ctx_.shared_owner == this) ctx_.shared_owner = nullptr;
    if (ctx_.static_owner == this) ctx_.static_owner = nullptr;
    for (hipEvent_t e : fork_events_)
        if (e != nullptr) (void)hipEventDestroy(e);
    for (auto &per_stage : join_events_)
        for (hipEvent_t e : per_stage)
            if (e != nullptr) (void)hipEventDestroy(e);
    for (hipEvent_t e : stage_events_) (void)hipEventDestroy(e);
    if (start_ != nullptr) (void)hipEventDestroy(start_);
    if (stop_ != nullptr) (void)hipEventDestroy(stop_);
    if (owns_memory_ && fused_items_ != nullptr) (void)hipFree(fused_items_);
    if (owns_memory_ && base_ != nullptr) (void)hipFree(base_);
    fork_events_.clear();
    join_events_.clear();
    stage_events_.clear();
    start_ = stop_ = nullptr;
    fused_items_ = nullptr;
    base_ = nullptr;
    if (!released_ && --ctx_.sessions == 0) ctx_.stage().give_back();   // (pinned memory for inputs and weights: up to 256 MB each)
    released_ = true;
}

TensorView Session::tv(const ViewRef &v) const {
    TensorView t;
    t.ptr = base_ + v.base + v.first;
    t.C = v.C;
    t.H = v.H;
    t.W = v.W;
    t.pstride = v.pstride;
    return t;
}

void Session::pack(const PlanConv &conv, hipStream_t stream) {
    if (conv.matrix_path) launch_pack_filters(conv.problem, conv.launch, base_ + conv.weight_off, base_ + conv.packed_off, stream);
    else if (conv.problem.is_depthwise()) launch_pack_depthwise(conv.problem, base_ + conv.weight_off, base_ + conv.packed_off, stream);
    packed_[&conv - plan_.convs.data()] = 1;
}

void Session::setup(bool pack_filters) {
    hipStream_t main = ctx_.stream(0);
    // (also where the memory is shared: a probe before this one left its tensors there)
    if (owns_memory_ || pack_filters) launch_fill_pattern(base_, plan_.arena_floats, 0x2468aceu, main);
    packed_.assign(plan_.convs.size(), 0);
    for (const PlanConv &conv : plan_.convs) {
        // A latency is measured without weights: filters with which the tensors neither grow from layer to layer nor with the sums
        // between them (half of He's bound; the biases of +-1 keep them from vanishing).  With +-1 they grow past 2^26 within five layers and
        // on to infinity, and sums of infinities are computed twice where two-term kernels meet them: no network's time.
        if (pack_filters)
            launch_fill_pattern(base_ + conv.weight_off, (size_t)conv.problem.OC * conv.problem.K(), 0x2468aceu, main, 0.5f * std::sqrt(6.f / (float)conv.problem.K()));
        // a convolution in front of the average pool it was exchanged with adds zeros; the pool adds the bias
        if (conv.linear) launch_fill_u32(reinterpret_cast<unsigned *>(base_ + conv.zero_bias_off), (size_t)conv.problem.OC, 0u, main);
        // split-K tickets start at zero; every launch leaves them at zero again
        if (conv.matrix_path && conv.ctr_count > 0) launch_fill_u32(reinterpret_cast<unsigned *>(base_ + conv.ctr_off), conv.ctr_count, 0u, main);
    }
    if (pack_filters) finish_weights();
}

void Session::finish_weights() {
    for (size_t c = 0; c < plan_.convs.size(); c++)
        if (!packed_[c]) pack(plan_.convs[c], ctx_.stream(0));
}

// events of the stream executors, created when the first pass needs them (a static session creates none)
void Session::ensure_fork_events() {
    const size_t num_stages = plan_.stages.size();
    if (fork_events_.size() == num_stages) return;
    fork_events_.assign(num_stages, nullptr);
    join_events_.assign(num_stages, {});
    for (size_t s = 0; s < num_stages; s++) {
        const size_t groups = plan_.stages[s].size();
        if (groups <= 1) continue;
        IOS_HIP(hipEventCreateWithFlags(&fork_events_[s], hipEventDisableTiming));
        join_events_[s].assign(groups - 1, nullptr);
        for (hipEvent_t &e : join_events_[s]) IOS_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    }
}

void Session::ensure_timers() {
    if (start_ == nullptr) IOS_HIP(hipEventCreate(&start_));
    if (stop_ == nullptr) IOS_HIP(hipEventCreate(&stop_));
}

void Session::set_input(const float *host) {
    if (host == nullptr) throw std::runtime_error("input pointer is null");
    const TensorView in = tv(plan_.input);
    hipStream_t main = ctx_.stream(0);
    input_changed_ = true;
    if (plan_.prefix_stages > 0) {
        // the first stages of the next pass start on the images that are there while the others are still on their way
        const size_t image = plan_.input.image_floats() * sizeof(float);
        arriving_.clear();
        std::vector<size_t> ends;
        for (int end : plan_.part_ends) ends.push_back(end * image);
        ctx_.stage().upload_chunks(base_ + plan_.landing_off, host, ends, ctx_.stream(1), main);
        arriving_ = plan_.part_ends;
        return;
    }
    arriving_.clear();
    ctx_.stage().upload_images(in, plan_.batch, host, main);
}

// images that have landed in the host's layout, the last of them with `chunk`, go to their place
void Session::take_images(int first, int images, int chunk) {
    hipStream_t main = ctx_.stream(0);
    ctx_.stage().arrived(chunk, main);
    TensorView in = tv(plan_.input);
    in.ptr += (size_t)first * in.H * in.W * in.pstride;
    launch_to_view(base_ + plan_.landing_off + (size_t)first * plan_.input.image_floats(), in, images, main);
}

// everything the next kernels of the main stream may read has arrived
void Session::settle() {
    if (!arriving_.empty()) take_images(0, plan_.batch, (int)arriving_.size() - 1);
    arriving_.clear();
}

// Filters and biases lie next to each other in the arena (the planner reserves them first, in network order): they are gathered
// by several threads and travel in large steps, on a stream of their own; the filters of a convolution are packed on the main
// stream as soon as they have arrived.
void Session::set_conv_weights(int count, char **names, float **weights, float **biases) {
    input_changed_ = true;
    std::vector<int> entry(plan_.convs.size(), -1);   // a name given twice: the last one counts
    for (int i = 0; i < count; i++) {
        auto it = plan_.conv_index.find(names[i] ? names[i] : "");
        if (it == plan_.conv_index.end()) {
            printf("%s not found\n", names[i] ? names[i] : "(null)");
            continue;
        }
        if (weights[i] == nullptr || biases[i] == nullptr)
            throw std::runtime_error(std::string("convolution '") + names[i] + "': weight or bias pointer is null");
        entry[it->second] = i;
    }
    std::vector<int> order;
    for (size_t c = 0; c < entry.size(); c++)
        if (entry[c] >= 0) order.push_back((int)c);
    std::sort(order.begin(), order.end(), [&](int a, int b) { return plan_.convs[a].weight_off < plan_.convs[b].weight_off; });
    std::vector<HostStage::Piece> pieces;
    std::vector<size_t> complete;   // per entry of `order`: the piece behind its bias
    auto add = [&](size_t offset, size_t floats, const float *src) {
        const size_t bytes = floats * sizeof(float);
        for (size_t at = 0; at < bytes; at += HostCopier::kPiece)
            pieces.push_back({offset * sizeof(float) + at, std::min(HostCopier::kPiece, bytes - at), reinterpret_cast<const char *>(src) + at});
    };
    for (int c : order) {   // (a filter lies in front of its bias)
        const PlanConv &conv = plan_.convs[c];
        add(conv.weight_off, (size_t)conv.problem.OC * conv.problem.K(), weights[entry[c]]);
        add(conv.bias_off, (size_t)conv.problem.OC, biases[entry[c]]);
        complete.push_back(pieces.size());
    }
    size_t next = 0;
    hipStream_t main = ctx_.stream(0);
    ctx_.stage().upload_pieces(reinterpret_cast<char *>(base_), pieces, ctx_.stream(1), main, [&](size_t limit) {
        for (; next < order.size() && complete[next] <= limit; next++) pack(plan_.convs[order[next]], main);
        if (advance_) advance();
    });
}

// Dense copy of a view in the host's layout.
void Session::copy_out(const ViewRef &view, float *host) {
    settle();
    ctx_.stage().download(host, tv(view), plan_.batch, ctx_.stream(0));
}

void Session::get_output(float *host) {
    if (host == nullptr) throw std::runtime_error("output pointer is null");
    if (!plan_.output_single_group) throw std::runtime_error("the last stage of the schedule must have a single group");
    fetches_result_ = true;
    if (ctx_.result_owner == this) ctx_.stage().fetch(host, (size_t)plan_.batch * plan_.output.image_floats() * sizeof(float), delivered_pass_, ctx_.stream(0));
    else copy_out(plan_.output, host);
}

void Session::get_tensor(const std::string &name, float *host) {
    auto it = plan_.tensors.find(name);
    if (it == plan_.tensors.end()) throw std::runtime_error("operator '" + name + "' has no materialised output");
    if (plan_.overwritten.count(name))
        throw std::runtime_error("the output of operator '" + name + "' shares its memory with a later operator and does not survive the pass "
                                 "(option arena_reuse=0 keeps every output)");
    if (ran_in_parts_ && plan_.in_parts.count(name)) {   // never whole in that pass: the same pass on the whole batch
        if (input_changed_)
            throw std::runtime_error("the last pass worked on parts of the batch, held the output of operator '" + name + "' for one part at a time, and its "
                                     "input or weights have changed since (option arena_reuse=0 keeps every output)");
        forward();
        synchronize();
    }
    copy_out(it->second, host);
}

unsigned *Session::counters_of(const PlanConv &c) const {
    if (c.ctr_count == 0 || !ctx_.inline_reduce()) return nullptr;
    return reinterpret_cast<unsigned *>(base_ + c.ctr_off);
}

// the images that a launch works on
TensorView Session::part_of(const ViewRef &whole_view, const ViewRef &part_view, bool whole, int first, int images) const {
    if (images <= 0) return tv(whole_view);
    TensorView t = tv(part_view);
    if (whole) t.ptr += (long long)first * t.H * t.W * t.pstride;
    return t;
}

void Session::launch_batch(const PlanBatch &batch, int first, int images) {
    ConvBatchMember members[kMaxConvBatch];
    int count = 0;
    MixedPool pool{};
    for (int index : batch.ops) {
        const PlanOp &op = plan_.ops[index];
        if (op.kind == OpKind::Pool) {
            pool = {op.pool, part_of(op.in, op.part_in, op.part_in_whole, first, images), part_of(op.out, op.part_out, op.part_out_whole, first, images),
                    op.bias_conv >= 0 ? base_ + plan_.convs[op.bias_conv].bias_off : nullptr, op.act};
            if (images > 0) pool.p.B = images;
            continue;
        }
        const PlanConv &c = plan_.convs[op.conv];
        ConvBatchMember &m = members[count++];
        m.p = c.problem;
        if (images > 0) m.p.B = images;
        m.packed = base_ + c.packed_off;
        m.filters = base_ + c.weight_off;
        m.bias = bias_of(c);
        m.y = part_of(op.out, op.part_out, op.part_out_whole, first, images);
        m.x = part_of(op.in, op.part_in, op.part_in_whole, first, images);
    }
    if (batch.mixed) launch_conv_mixed(members, count, pool.x.ptr != nullptr ? &pool : nullptr, batch.variant, ctx_.stream(0));
    else launch_conv_batch(members, count, batch.variant, ctx_.stream(0));
}

void Session::launch_batches(size_t stage, int first, int images) {
    for (const PlanBatch &batch : plan_.batches)
        if (batch.stage == (int)stage) launch_batch(batch, first, images);
}

// The same where the stages are timed: what a batch would take ahead runs in the stage that the schedule gives it, by itself.
void Session::launch_scheduled_batches(size_t stage) {
    for (const PlanBatch &batch : plan_.batches) {
        if (!batch.across_stages) {
            if (batch.stage == (int)stage) launch_batch(batch);
            continue;
        }
        for (int op : batch.ops)
            if (plan_.ops[op].scheduled_stage() == (int)stage) launch_op(plan_.ops[op], 0);
    }
}

void Session::launch_op(const PlanOp &op, int group, int first, int images) {
    hipStream_t stream = ctx_.stream(group);
    const int count = images > 0 ? images : plan_.batch;
    const TensorView in = part_of(op.in, op.part_in, op.part_in_whole, first, images), out = part_of(op.out, op.part_out, op.part_out_whole, first, images);
    switch (op.kind) {
        case OpKind::ConvMfma: {
            const PlanConv &c = plan_.convs[op.conv];
            ConvProblem p = c.problem;
            p.B = count;
            const TensorView residual = op.has_residual ? tv(op.residual) : TensorView{};
            launch_conv_mfma(p, c.launch, in, base_ + c.packed_off, base_ + c.weight_off, bias_of(c), out,
                             c.ws_floats ? base_ + c.ws_off : nullptr, ctx_.split_reduce(counters_of(c), group, !capturing_forks_), stream,
                             op.has_residual ? &residual : nullptr,
                             op.post_relu != 0);
            break;
        }
        case OpKind::ConvDepthwise: {
            const PlanConv &c = plan_.convs[op.conv];
            ConvProblem p = c.problem;
            p.B = count;
            TensorView more[kMaxNaryInputs];
            for (size_t i = 1; i < op.srcs.size(); i++) more[i - 1] = tv(op.srcs[i]);
            launch_dwconv(p, in, base_ + c.packed_off, bias_of(c), out, stream, more,
                          op.srcs.empty() ? 0 : (int)op.srcs.size() - 1);
            break;
        }
        case OpKind::ConvDirect: {
            const PlanConv &c = plan_.convs[op.conv];
            ConvProblem p = c.problem;
            p.B = count;
            launch_conv_direct(p, in, base_ + c.weight_off, bias_of(c), out, stream, c.thin);
            break;
        }
        case OpKind::Pool:
        case OpKind::GlobalPool: {
            PoolProblem p = op.pool;
            p.B = count;
            if (op.kind == OpKind::GlobalPool) launch_global_pool(p, in, out, stream);
            else launch_pool(p, in, out, stream, op.bias_conv >= 0 ? base_ + plan_.convs[op.bias_conv].bias_off : nullptr, op.act);
            break;
        }
        case OpKind::Nary: {
            NaryArgs a;
            a.count = (int)op.srcs.size();
            for (int i = 0; i < a.count; i++) {
                a.src[i] = tv(op.srcs[i]).ptr;
                a.src_pstride[i] = op.srcs[i].pstride;
            }
            launch_nary(a, op.multiply, op.accumulate, op.act, count, out, stream);
            break;
        }
        case OpKind::Unary: launch_unary(in, out, op.act, count, stream); break;
    }
}

void Session::enqueue_stage_streams(size_t s) {
    hipStream_t main = ctx_.stream(0);
    const auto &groups = plan_.stages[s];
    const bool fork = groups.size() > 1;
    if (fork) {
        IOS_HIP(hipEventRecord(fork_events_[s], main));
        for (size_t g = 1; g < groups.size(); g++) IOS_HIP(hipStreamWaitEvent(ctx_.stream((int)g), fork_events_[s], 0));
    }
    for (size_t g = 0; g < groups.size(); g++)
        for (int op : groups[g]) launch_op(plan_.ops[op], (int)g);
    if (fork) {
        for (size_t g = 1; g < groups.size(); g++) {
            IOS_HIP(hipEventRecord(join_events_[s][g - 1], ctx_.stream((int)g)));
            IOS_HIP(hipStreamWaitEvent(main, join_events_[s][g - 1], 0));
        }
    }
}

void Session::enqueue_stage_serial(size_t s) {
    for (const auto &group : plan_.stages[s])
        for (int op : group) launch_op(plan_.ops[op], 0);
}

void Session::enqueue_stage(size_t s, bool timed) {
    if (timed) launch_scheduled_batches(s);
    else launch_batches(s);
    if (static_) enqueue_stage_serial(s);
    else if (ctx_.fused_executor()) enqueue_stage_fused(s);
    else enqueue_stage_streams(s);
}

// what enqueue_stage needs beyond the plan: allocations, copies and events stay outside a graph capture
void Session::ready_executor() {
    if (static_) return;
    if (ctx_.fused_executor()) build_fused();
    else ensure_fork_events();
}

// issues the stages from `first` on in order
void Session::enqueue(size_t first, bool stage_events) {
    if (static_ && stage_events) throw std::runtime_error("a session in the static scratch cannot profile stages");
    ready_executor();
    for (size_t s = first; s < plan_.stages.size(); s++) {
        enqueue_stage(s, stage_events);
        if (stage_events) IOS_HIP(hipEventRecord(stage_events_[s], ctx_.stream(0)));
    }
}

// The leading stages, of one group each: on the whole batch, or part by part as the images arrive.
void Session::enqueue_prefix(size_t stages) {
    input_changed_ = false;
    ran_in_parts_ = !arriving_.empty() && plan_.prefix_stages > 0;
    if (!ran_in_parts_) {
        settle();
        for (size_t s = 0; s < stages; s++) enqueue_stage(s);
        return;
    }
    const size_t split = (size_t)plan_.prefix_stages;
    int begin = 0;
    // (a part's stages follow those of the part before it: they write over the tensors that hold one part at a time)
    for (size_t part = 0; part < arriving_.size(); part++) {
        const int images = arriving_[part] - begin;
        take_images(begin, images, (int)part);
        for (size_t s = 0; s < split; s++) {
            launch_batches(s, begin, images);
            for (int op : plan_.stages[s][0]) launch_op(plan_.ops[op], 0, begin, images);
        }
        begin = arriving_[part];
    }
    arriving_.clear();
    for (size_t s = split; s < stages; s++) enqueue_stage(s);
}

// ---- fused stage launches -----------------------------------------------------------------------------------------
// A stage is cut into levels: the operations of a group follow each other, except that operations of one unit on the same
// PlanOp::level (the terms of a concatenation) share a level; a split-K convolution contributes its main kernel and, with
// the two-kernel reduction, one level later its reduction.  The kernels of one level are independent and become work items
// of one fused launch; levels follow each other on the main stream.  A single-group stage keeps its stand-alone kernels on
// the levels that hold one operation.
void Session::build_fused() {
    if (fused_built_) return;
    std::vector<WorkItem> items;
    fused_stages_.assign(plan_.stages.size(), {});
    struct Pending {
        WorkItem item;
        int threads;     // 0: any block size
        int smem_bytes;
        int op;          // plan operation behind the item
        bool fusable;
    };
    for (size_t s = 0; s < plan_.stages.size(); s++) {
        const auto &groups = plan_.stages[s];
        const bool solo = groups.size() <= 1;
        if (solo) {
            bool shared_level = false;
            for (const auto &group : groups)
                for (size_t i = 1; i < group.size(); i++) {
                    const PlanOp &a = plan_.ops[group[i - 1]], &b = plan_.ops[group[i]];
                    if (a.unit == b.unit && a.level == b.level) shared_level = true;
                }
            if (!shared_level) continue;
        }
        std::vector<std::vector<std::vector<Pending>>> chains(groups.size());   // group, level, items
        for (size_t g = 0; g < groups.size(); g++) {
            auto &chain = chains[g];
            int unit = -2;
            size_t base = 0, shift = 0;
            auto level_of = [&](const PlanOp &op) -> std::vector<Pending> & {
                if (op.unit != unit) {
                    unit = op.unit;
                    base = chain.size();
                    shift = 0;
                }
                const size_t at = base + shift + (size_t)op.level;
                if (chain.size() <= at) chain.resize(at + 1);
                return chain[at];
            };
            for (int index : groups[g]) {
                const PlanOp &op = plan_.ops[index];
                Pending pend;
                memset(&pend.item, 0, sizeof(WorkItem));
                pend.threads = 0;
                pend.smem_bytes = 0;
                pend.op = index;
                pend.fusable = true;
                int blocks = 0;
                switch (op.kind) {
                    case OpKind::ConvMfma: {
                        const PlanConv &c = plan_.convs[op.conv];
                        const TensorView residual = op.has_residual ? tv(op.residual) : TensorView{};
                        const ConvDispatch d = make_conv_dispatch(c.problem, c.launch, tv(op.in), base_ + c.packed_off, base_ + c.weight_off, bias_of(c),
                                                                  tv(op.out), c.ws_floats ? base_ + c.ws_off : nullptr, ctx_.split_reduce(counters_of(c)),
                                                                  op.has_residual ? &residual : nullptr, op.post_relu != 0);
                        pend.fusable = conv_variant(d.variant).fusable() && !op.has_residual;   // (the fused kernel holds the plain epilogue)
                        if (!pend.fusable && !solo && (op.has_residual || ctx_.forced_variant() >= 0))
                            throw std::runtime_error(op.has_residual ? std::string("internal: a residual convolution is planned for single-group stages only")
                                                                     : std::string("convolution kernel configuration ") + conv_variant(d.variant).name +
                                                                           " cannot run inside a fused stage launch");
                        pend.item = conv_work_item(d);
                        pend.threads = d.threads;
                        pend.smem_bytes = d.smem_bytes;
                        if (d.has_reduce && solo) pend.fusable = false;   // launched stand-alone, reduction included
                        level_of(op).push_back(pend);
                        if (d.has_reduce && pend.fusable) {
                            Pending red;
                            memset(&red.item, 0, sizeof(WorkItem));
                            red.item.kind = WORK_REDUCE;
                            red.item.num_blocks = d.reduce_blocks;
                            red.item.reduce = d.reduce;
                            red.threads = 0;
                            red.smem_bytes = 0;
                            red.op = index;
                            red.fusable = true;
                            shift++;
                            level_of(op).push_back(red);
                        }
                        continue;
                    }
                    case OpKind::ConvDepthwise:
                    case OpKind::ConvDirect: {
                        const PlanConv &c = plan_.convs[op.conv];
                        pend.item.kind = op.kind == OpKind::ConvDepthwise ? WORK_DWCONV : WORK_CONV_DIRECT;
                        if (c.thin) throw std::runtime_error("internal: the thin-input convolution kernel is planned for single-group stages only");
                        pend.item.direct = make_direct_conv_args(c.problem, tv(op.in), base_ + (op.kind == OpKind::ConvDepthwise ? c.packed_off : c.weight_off),
                                                                 bias_of(c), tv(op.out), &blocks);
                        if (op.kind == OpKind::ConvDepthwise && op.srcs.size() > 1) {
                            TensorView more[kMaxNaryInputs];
                            for (size_t i = 1; i < op.srcs.size(); i++) more[i - 1] = tv(op.srcs[i]);
                            add_dwconv_sources(pend.item.direct, more, (int)op.srcs.size() - 1, &blocks);
                        }
                        break;
                    }
                    case OpKind::Pool:
                    case OpKind::GlobalPool:
                        pend.item.kind = op.kind == OpKind::Pool ? WORK_POOL : WORK_GLOBAL_POOL;
                        pend.item.pool = make_pool_args(op.pool, tv(op.in), tv(op.out), op.kind == OpKind::GlobalPool, &blocks,
                                                        op.bias_conv >= 0 ? base_ + plan_.convs[op.bias_conv].bias_off : nullptr, op.act);
                        break;
                    case OpKind::Nary:
                    case OpKind::Unary: {
                        NaryArgs in;
                        if (op.kind == OpKind::Unary) {
                            in.count = 1;
                            in.src[0] = tv(op.in).ptr;
                            in.src_pstride[0] = op.in.pstride;
                        } else {
                            in.count = (int)op.srcs.size();
                            for (int i = 0; i < in.count; i++) {
                                in.src[i] = tv(op.srcs[i]).ptr;
                                in.src_pstride[i] = op.srcs[i].pstride;
                            }
                        }
                        pend.item.kind = WORK_NARY;
                        pend.item.nary = make_nary_args(in, op.multiply, op.accumulate, op.act, plan_.batch, tv(op.out), &blocks);
                        break;
                    }
                }
                pend.item.num_blocks = blocks;   // sized for 256-thread blocks, rescaled below
                level_of(op).push_back(pend);
            }
        }
        size_t depth = 0;
        for (const auto &chain : chains) depth = std::max(depth, chain.size());
        for (size_t level = 0; level < depth; level++) {
            std::vector<Pending *> here;
            int widest = 0;
            bool all_fusable = true;
            for (auto &chain : chains)
                if (level < chain.size())
                    for (Pending &pend : chain[level]) {
                        if (!solo && !pend.fusable) {   // fills the device by itself (see tune_conv); the others of the level share launches
                            fused_stages_[s].push_back(FusedLaunch{0, 0, 0, 0, 0, pend.op, {}, {pend.op}});
                            continue;
                        }
                        here.push_back(&pend);
                        widest = std::max(widest, pend.threads);
                        all_fusable = all_fusable && pend.fusable;
                    }
            if (here.empty()) continue;
            // a configuration of the wide-register family beside a 1024-thread body: that family has no such form, the
            // operators of the level are launched one after the other instead (they are independent of each other)
            bool needs_wide = false;
            for (Pending *pend : here)
                needs_wide = needs_wide || (pend->item.kind == WORK_CONV && conv_variant(pend->item.variant).needs_wide());
            if (needs_wide && widest > 512 && all_fusable) {
                for (Pending *pend : here)
                    if (pend->item.kind != WORK_REDUCE)   // (a stand-alone split-K launch brings its own reduction)
                        fused_stages_[s].push_back(FusedLaunch{0, 0, 0, 0, 0, pend->op, {}, {pend->op}});
                continue;
            }
            if (solo && (here.size() == 1 || !all_fusable)) {
                for (Pending *pend : here) fused_stages_[s].push_back(FusedLaunch{0, 0, 0, 0, 0, pend->op, {}, {pend->op}});
                continue;
            }
            widest = std::max(widest, 256);   // narrowest instantiation of the fused kernel
            // one launch per level, as wide as its widest convolution body; more items than a launch holds: several launches
            for (size_t first = 0; first < here.size(); first += kMaxFusedItems) {
                const size_t last = std::min(here.size(), first + (size_t)kMaxFusedItems);
                FusedLaunch launch{widest, (int)items.size(), 0, 0, 0, -1, {}, {}};
                for (size_t i = first; i < last; i++) {
                    Pending *pend = here[i];
                    launch.ops.push_back(pend->op);
                    WorkItem item = pend->item;
                    item.threads = pend->threads == 0 ? widest : pend->threads;
                    if (pend->threads == 0) item.num_blocks = std::max(1, (item.num_blocks * 256 + widest - 1) / widest);
                    item.first_block = launch.total_blocks;
                    if (launch.num_items < kFusedHeaderItems) launch.header.first_block[launch.num_items] = item.first_block;
                    launch.total_blocks += item.num_blocks;
                    launch.smem_bytes = std::max(launch.smem_bytes, pend->smem_bytes);
                    launch.num_items++;
                    items.push_back(item);
                }
                launch.header.num_items = launch.num_items;
                fused_stages_[s].push_back(launch);
            }
        }
    }
    fused_items_host_ = items;
    if (!items.empty()) {
        if (owns_memory_) IOS_HIP(hipMalloc(&fused_items_, items.size() * sizeof(WorkItem)));
        else fused_items_ = ctx_.shared_table(items.size() * sizeof(WorkItem));
        ctx_.stage().upload(fused_items_, items.data(), items.size() * sizeof(WorkItem), ctx_.stream(0));
    }
    fused_built_ = true;
}

void Session::enqueue_stage_fused(size_t s) {
    if (fused_stages_[s].empty()) {
        enqueue_stage_serial(s);
        return;
    }
    const WorkItem *items = static_cast<const WorkItem *>(fused_items_);
    for (const FusedLaunch &l : fused_stages_[s]) {
        if (l.single_op >= 0) launch_op(plan_.ops[l.single_op], 0);
        else launch_fused(l.threads, items + l.first_item, fused_items_host_.data() + l.first_item, l.header, l.total_blocks, l.smem_bytes, ctx_.num_cus(), ctx_.stream(0));
    }
}

// Leading stages that the graph executors launch directly.  Handing a graph to the device takes the host 14-22 us before its
// first kernel starts (measured for 1 to 60 kernels; a kernel launch takes 1.6-2.5 us), so the first few kernels go ahead of
// it and the device works on them meanwhile; a pass of a handful of kernels needs no graph at all.
size_t Session::direct_stages() const {
    constexpr size_t kAhead = 4, kNoGraph = 8;
    auto launches_of = [&](size_t s) {
        size_t ops = 0, batches = 0;
        for (const auto &group : plan_.stages[s]) ops += group.size();
        for (const PlanBatch &batch : plan_.batches) batches += batch.stage == (int)s ? 1 : 0;
        return batches + (ctx_.fused_executor() && !fused_stages_[s].empty() ? fused_stages_[s].size() : ops);
    };
    size_t total = 0, ahead = 0, stages = 0;
    for (size_t s = 0; s < plan_.stages.size(); s++) total += launches_of(s);
    if (ctx_.fused_executor() && total <= kNoGraph) return plan_.stages.size();
    while (stages < plan_.stages.size() && ahead < kAhead) {
        if (!ctx_.fused_executor() && plan_.stages[stages].size() > 1) break;
        ahead += launches_of(stages++);
    }
    return std::max(stages, (size_t)plan_.prefix_stages);
}

void Session::build_graph(size_t first) {
    hipStream_t main = ctx_.stream(0);
    IOS_HIP(hipStreamBeginCapture(main, hipStreamCaptureModeRelaxed));
    // the stream executor forks inside the capture, and the replay runs the branches on streams of its own choice
    capturing_forks_ = ctx_.exec_mode() == ExecMode::Graph;
    try {
        enqueue(first, false);
        capturing_forks_ = false;
    } catch (...) {
        capturing_forks_ = false;
        hipGraph_t broken = nullptr;
        (void)hipStreamEndCapture(main, &broken);
        if (broken != nullptr) (void)hipGraphDestroy(broken);
        throw;
    }
    IOS_HIP(hipStreamEndCapture(main, &graph_));
    IOS_HIP(hipGraphInstantiate(&graph_exec_, graph_, nullptr, nullptr, 0));
}

void Session::drop_graph() noexcept {
    if (graph_exec_ != nullptr) (void)hipGraphExecDestroy(graph_exec_);
    if (graph_ != nullptr) (void)hipGraphDestroy(graph_);
    graph_exec_ = nullptr;
    graph_ = nullptr;
}

void Session::forward() {
    if (ctx_.result_owner == this) ctx_.result_owner = nullptr;
    ready_executor();
    const ExecMode mode = ctx_.exec_mode();
    if (static_ || (mode != ExecMode::Graph && mode != ExecMode::FusedGraph)) {
        const size_t prefix = (size_t)plan_.prefix_stages;
        enqueue_prefix(prefix);
        enqueue(prefix, false);
        return;
    }
    const size_t direct = direct_stages();
    if (graph_exec_ != nullptr && graph_mode_ != mode) drop_graph();   // the option changed since the capture
    if (graph_exec_ == nullptr && direct < plan_.stages.size()) {
        build_graph(direct);
        graph_mode_ = mode;
    }
    enqueue_prefix(direct);
    if (direct < plan_.stages.size()) IOS_HIP(hipGraphLaunch(graph_exec_, ctx_.stream(0)));
}

void Session::run() {
    forward();
    finish_pass();
}

// waits for the pass that was queued last
void Session::finish_pass() {
    // A result of a few pages costs the last kernel nothing; a larger one travels with the pass unless the caller has left the
    // one before where it was (it is then copied when it is asked for).
    constexpr size_t kAlways = size_t(64) << 10;
    const size_t bytes = (size_t)plan_.batch * plan_.output.image_floats() * sizeof(float);
    const bool deliver = plan_.output_single_group && (bytes <= kAlways || (fetches_result_ && bytes <= HostStage::kResult));
    fetches_result_ = false;
    HostStage::Result result;
    if (deliver) result = {tv(plan_.output), plan_.batch};
    hipStream_t main = ctx_.stream(0);
    if (deliver) ctx_.result_owner = nullptr;   // what is there is written over, also by a pass that then fails
    const unsigned pass = ctx_.stage().signal(result, main);
    ctx_.stage().wait(pass, main);
    ctx_.check_xcd_fault();
    if (!deliver) return;
    ctx_.result_owner = this;
    delivered_pass_ = pass;
}

// One inference with everything crossing the boundary.  The weights of a network take longer on the link than the pass itself
// (87 MB, 1.5 ms against 0.4 ms for Inception-v3 at batch 1), so a stage is issued as soon as the filters of its convolutions
// have been: the pass runs behind the transfer and ends with the stages of the last part.
void Session::infer(const float *input, int count, char **names, float **weights, float **biases, float *output) {
    attach();
    if (ctx_.result_owner == this) ctx_.result_owner = nullptr;
    set_input(input);
    settle();
    ready_executor();
    packed_.assign(plan_.convs.size(), 0);
    next_stage_ = 0;
    advance_ = true;
    try {
        set_conv_weights(count, names, weights, biases);
        finish_weights();
        advance();
    } catch (...) {
        advance_ = false;
        throw;
    }
    advance_ = false;
    fetches_result_ = true;
    finish_pass();
    get_output(output);
}

// issues the stages whose filters are packed
void Session::advance() {
    for (; next_stage_ < plan_.stages.size(); next_stage_++) {
        for (const PlanBatch &batch : plan_.batches)
            if (batch.stage == (int)next_stage_)
                for (int op : batch.ops) {
                    const int conv = plan_.ops[op].conv >= 0 ? plan_.ops[op].conv : plan_.ops[op].bias_conv;
                    if (conv >= 0 && !packed_[conv]) return;
                }
        for (const auto &group : plan_.stages[next_stage_])
            for (int op : group)
                if (plan_.ops[op].conv >= 0 && !packed_[plan_.ops[op].conv]) return;
        for (const auto &group : plan_.stages[next_stage_])
            for (int op : group)
                if (plan_.ops[op].bias_conv >= 0 && !packed_[plan_.ops[op].bias_conv]) return;
        enqueue_stage(next_stage_);
    }
}

// A session in memory that others use in between (the shared arena, the static scratch) lays out again what it keeps there.
void Session::attach() {
    if (owns_memory_) return;
    float *base = static_ ? ctx_.static_scratch() : ctx_.shared_arena(plan_.arena_floats);
    const void *&owner = static_ ? ctx_.static_owner : ctx_.shared_owner;
    if (base == base_ && owner == this) return;
    base_ = base;
    owner = this;
    drop_graph();
    fused_built_ = false;
    setup(false);
}

void Session::synchronize() {
    IOS_HIP(hipStreamSynchronize(ctx_.stream(0)));
    ctx_.check_xcd_fault();
}

void Session::measure(int warmup, int number, int repeat, bool profile_stage, float *results, float *stage_results) {
    if (static_) throw std::runtime_error("a session in the static scratch has no timers");
    if (number < 1 || repeat < 1 || warmup < 0) throw std::runtime_error("measure: warmup >= 0, number >= 1, repeat >= 1 required");
    ensure_timers();
    hipStream_t main = ctx_.stream(0);
    const size_t num_stages = plan_.stages.size();
    if (profile_stage && stage_events_.empty()) {
        stage_events_.resize(num_stages);
        for (hipEvent_t &e : stage_events_) IOS_HIP(hipEventCreate(&e));
    }
    auto pass = [&]() {
        if (profile_stage) {
            settle();
            ran_in_parts_ = input_changed_ = false;
            enqueue(0, true);
        }
        else forward();
    };
    for (int i = 0; i < warmup; i++) pass();
    for (int i = 0; i < repeat; i++) {
        double total = 0.0;
        std::vector<double> per_stage(num_stages, 0.0);
        for (int t = 0; t < number; t++) {
            IOS_HIP(hipDeviceSynchronize());
            IOS_HIP(hipEventRecord(start_, main));
            pass();
            IOS_HIP(hipEventRecord(stop_, main));
            IOS_HIP(hipEventSynchronize(stop_));
            float ms = 0.f;
            if (profile_stage) {
                for (size_t s = 0; s < num_stages; s++) {
                    hipEvent_t from = s == 0 ? start_ : stage_events_[s - 1];
                    hipEvent_t to = s + 1 == num_stages ? stop_ : stage_events_[s];
                    IOS_HIP(hipEventElapsedTime(&ms, from, to));
                    per_stage[s] += ms;
                }
            }
            IOS_HIP(hipEventElapsedTime(&ms, start_, stop_));
            total += ms;
        }
        results[i] = (float)(total / number);
        if (profile_stage && stage_results != nullptr)
            for (size_t s = 0; s < num_stages; s++) stage_results[i * num_stages + s] = (float)(per_stage[s] / number);
    }
    IOS_HIP(hipDeviceSynchronize());
    ctx_.check_xcd_fault();
}

void Session::measure_back_to_back(int warmup, int number, int repeat, float *results) {
    if (static_) throw std::runtime_error("a session in the static scratch has no timers");
    if (number < 1 || repeat < 1 || warmup < 0) throw std::runtime_error("measure: warmup >= 0, number >= 1, repeat >= 1 required");
    ensure_timers();
    hipStream_t main = ctx_.stream(0);
    for (int i = 0; i < warmup; i++) forward();
    for (int i = 0; i < repeat; i++) {
        IOS_HIP(hipDeviceSynchronize());
        IOS_HIP(hipEventRecord(start_, main));
        for (int t = 0; t < number; t++) forward();
        IOS_HIP(hipEventRecord(stop_, main));
        IOS_HIP(hipEventSynchronize(stop_));
        float ms = 0.f;
        IOS_HIP(hipEventElapsedTime(&ms, start_, stop_));
        results[i] = ms / (float)number;
    }
    IOS_HIP(hipDeviceSynchronize());
    ctx_.check_xcd_fault();
}

void Session::profile_ops(int warmup, int repeat, float *ms_out) {
    if (static_) throw std::runtime_error("a session in the static scratch has no timers");
    if (repeat < 1 || warmup < 0) throw std::runtime_error("profile_ops: warmup >= 0 and repeat >= 1 required");
    ensure_timers();
    hipStream_t main = ctx_.stream(0);
    settle();
    run();   // every operator sees the inputs it has in a real pass, on the whole batch
    for (size_t i = 0; i < plan_.ops.size(); i++) {
        const PlanOp &op = plan_.ops[i];
        for (int w = 0; w < warmup; w++) launch_op(op, 0);
        IOS_HIP(hipStreamSynchronize(main));
        IOS_HIP(hipEventRecord(start_, main));
        for (int r = 0; r < repeat; r++) launch_op(op, 0);
        IOS_HIP(hipEventRecord(stop_, main));
        IOS_HIP(hipEventSynchronize(stop_));
        float ms = 0.f;
        IOS_HIP(hipEventElapsedTime(&ms, start_, stop_));
        ms_out[i] = ms / (float)repeat;
    }
}

// ---- per-launch view of a pass -------------------------------------------------------------------------------------------
static std::string op_kernel_name(const Plan &plan, const PlanOp &op) {
    switch (op.kind) {
        case OpKind::ConvMfma: return std::string("conv_kernel<") + conv_variant(plan.convs[op.conv].launch.variant).name + ">";
        case OpKind::ConvDepthwise: return "dwconv_kernel";
        case OpKind::ConvDirect: return plan.convs[op.conv].thin ? "conv_thin_kernel" : "conv_direct_kernel";
        case OpKind::Pool: return "pool_kernel";
        case OpKind::GlobalPool: return "global_pool_kernel";
        case OpKind::Nary:
        case OpKind::Unary: return "nary_kernel";
    }
    return "?";
}

std::vector<Session::LaunchRecord> Session::launches() {
    const ExecMode mode = ctx_.exec_mode();
    const bool fused = !static_ && (mode == ExecMode::Fused || mode == ExecMode::FusedGraph);
    if (fused) build_fused();
    std::vector<LaunchRecord> out;
    for (size_t s = 0; s < plan_.stages.size(); s++) {
        const auto &groups = plan_.stages[s];
        for (size_t b = 0; b < plan_.batches.size(); b++) {
            if (plan_.batches[b].stage != (int)s) continue;
            LaunchRecord r;
            r.stage = (int)s;
            r.kernel = std::string(plan_.batches[b].mixed ? "conv_mixed_kernel<" : "conv_batch_kernel<") + conv_variant(plan_.batches[b].variant).name + ">";
            r.ops = plan_.batches[b].ops;
            r.batch = (int)b;
            out.push_back(r);
        }
        if (fused && !fused_stages_[s].empty()) {
            for (size_t l = 0; l < fused_stages_[s].size(); l++) {
                const FusedLaunch &f = fused_stages_[s][l];
                LaunchRecord r;
                r.stage = (int)s;
                if (f.single_op >= 0) {
                    r.kernel = op_kernel_name(plan_, plan_.ops[f.single_op]);
                    r.ops = {f.single_op};
                    out.push_back(r);
                    continue;
                }
                const FusedForm form = fused_launch_form(fused_items_host_.data() + f.first_item, f.num_items, f.threads, f.total_blocks, ctx_.num_cus());
                r.kernel = std::string(fused_kernel_name(form)) + "<" + std::to_string(f.threads) + ">";
                r.ops = f.ops;
                r.blocks = f.total_blocks;
                r.threads = f.threads;
                r.fused_level = (int)l;
                out.push_back(r);
            }
            continue;
        }
        for (const auto &group : groups)
            for (int index : group) {
                LaunchRecord r;
                r.stage = (int)s;
                r.kernel = op_kernel_name(plan_, plan_.ops[index]);
                r.ops = {index};
                out.push_back(r);
            }
    }
    return out;
}

std::string Session::describe_launches() {
    std::ostringstream os;
    os << '[';
    bool first = true;
    for (const LaunchRecord &r : launches()) {
        double flops = 0.0, bytes = 0.0, conv_flops = 0.0;
        std::vector<int> seen;
        for (int index : r.ops) {
            if (std::find(seen.begin(), seen.end(), index) != seen.end()) continue;
            seen.push_back(index);
            flops += plan_.ops[index].flops;
            bytes += plan_.ops[index].bytes;
            if (plan_.ops[index].kind == OpKind::ConvMfma) conv_flops += plan_.ops[index].flops;
        }
        os << (first ? "" : ",") << "{\"stage\":" << r.stage << ",\"kernel\":\"" << r.kernel << "\",\"fused_level\":" << r.fused_level
           << ",\"blocks\":" << r.blocks << ",\"threads\":" << r.threads << ",\"flops\":" << flops << ",\"matrix_flops\":" << conv_flops
           << ",\"bytes\":" << bytes << ",\"ops\":[";
        for (size_t i = 0; i < seen.size(); i++) os << (i ? "," : "") << seen[i];
        os << "]}";
        first = false;
    }
    os << ']';
    return os.str();
}

void Session::profile_launches(int warmup, int repeat, float *ms_out, int capacity) {
    if (static_) throw std::runtime_error("a session in the static scratch has no timers");
    if (repeat < 1 || warmup < 0) throw std::runtime_error("profile_launches: warmup >= 0 and repeat >= 1 required");
    const std::vector<LaunchRecord> list = launches();
    if ((int)list.size() > capacity) throw std::runtime_error("profile_launches: output array too small");
    ensure_timers();
    hipStream_t main = ctx_.stream(0);
    settle();
    run();   // every launch sees the inputs it has in a real pass, on the whole batch
    const WorkItem *items = static_cast<const WorkItem *>(fused_items_);
    for (size_t i = 0; i < list.size(); i++) {
        const LaunchRecord &r = list[i];
        auto issue = [&]() {
            if (r.batch >= 0) {
                launch_batch(plan_.batches[r.batch]);
            } else if (r.fused_level >= 0) {
                const FusedLaunch &l = fused_stages_[r.stage][r.fused_level];
                launch_fused(l.threads, items + l.first_item, fused_items_host_.data() + l.first_item, l.header, l.total_blocks, l.smem_bytes, ctx_.num_cus(), main);
            } else {
                launch_op(plan_.ops[r.ops[0]], 0);
            }
        };
        for (int w = 0; w < warmup; w++) issue();
        IOS_HIP(hipStreamSynchronize(main));
        IOS_HIP(hipEventRecord(start_, main));
        for (int k = 0; k < repeat; k++) issue();
        IOS_HIP(hipEventRecord(stop_, main));
        IOS_HIP(hipEventSynchronize(stop_));
        float ms = 0.f;
        IOS_HIP(hipEventElapsedTime(&ms, start_, stop_));
        ms_out[i] = ms / (float)repeat;
    }
}

}  // namespace ios
