#include "host_io.h"

#include <algorithm>
#include <chrono>
#include <climits>
#include <cstring>
#include <stdexcept>
#include <thread>

#include <linux/futex.h>
#include <sys/syscall.h>
#include <unistd.h>
#if defined(__x86_64__)
#include <emmintrin.h>
#endif

#include "runtime.h"

namespace ios {

// ---- threads -----------------------------------------------------------------------------------------------------------
HostCopier &HostCopier::get() {
    static HostCopier *instance = new HostCopier();
    return *instance;
}

static inline void pause() {
#if defined(__x86_64__)
    __builtin_ia32_pause();
#endif
}

void HostCopier::rouse() {
    if (!started_) start();
    calls_.fetch_add(1);
    syscall(SYS_futex, reinterpret_cast<unsigned *>(&calls_), FUTEX_WAKE_PRIVATE, 3, nullptr, nullptr, 0);
}

void HostCopier::start() {
    started_ = true;
    // half of the processors this process may use, eight at most: past that the copies are bound by memory, not by threads
    const int n = std::min(8, std::max(1, (int)std::thread::hardware_concurrency() / 2));
    for (int i = 1; i < n; i++) std::thread([this]() { worker(); }).detach();
}

void HostCopier::worker() {
    unsigned seen = 0, heard = 0;
    for (;;) {
        const unsigned call = calls_.load();
        unsigned now = generation_.load();
        if (now == seen && call == heard) {
            syscall(SYS_futex, reinterpret_cast<unsigned *>(&calls_), FUTEX_WAIT_PRIVATE, call, nullptr, nullptr, 0);
            continue;
        }
        heard = call;
        if (now == seen) {   // roused
            const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(1);
            while ((now = generation_.load()) == seen && std::chrono::steady_clock::now() < until)
                for (int i = 0; i < 16; i++) pause();
            if (now == seen) continue;
        }
        seen = now;
        // either the owner sees this thread in busy_ and waits for it, or this thread sees that the copy is closed
        busy_.fetch_add(1);
        if (open_.load() == now)
            for (int i; (i = next_.fetch_add(1)) < pieces_;) (*body_)(i);
        busy_.fetch_sub(1);
    }
}

void HostCopier::parallel(int pieces, const std::function<void(int)> &body, const std::function<void()> *idle) {
    if (pieces <= 1) {
        if (pieces == 1) body(0);
        if (idle != nullptr) (*idle)();
        return;
    }
    if (!started_) start();
    next_.store(0);
    body_ = &body;
    pieces_ = pieces;
    unsigned generation = generation_.load() + 1;
    if (generation == 0) generation = 1;
    open_.store(generation);
    generation_.store(generation);
    calls_.fetch_add(1);
    syscall(SYS_futex, reinterpret_cast<unsigned *>(&calls_), FUTEX_WAKE_PRIVATE, INT_MAX, nullptr, nullptr, 0);
    for (int i; (i = next_.fetch_add(1)) < pieces;) {
        body(i);
        if (idle != nullptr) (*idle)();
    }
    open_.store(0);
    while (busy_.load() != 0) {
        if (idle != nullptr) (*idle)();
        pause();
    }
    if (idle != nullptr) (*idle)();
}

void HostCopier::copy(void *dst, const void *src, size_t bytes) {
    if (bytes < kParallelBytes) {
        memcpy(dst, src, bytes);
        return;
    }
    parallel((int)((bytes + kPiece - 1) / kPiece), [&](int i) {
        const size_t at = (size_t)i * kPiece;
        memcpy(static_cast<char *>(dst) + at, static_cast<const char *>(src) + at, std::min(kPiece, bytes - at));
    });
}

// Fills a buffer that only the link will read and that is larger than the caches: stores past the caches save reading every
// line of the buffer first (a third of the copy's memory traffic).
static void copy_past_caches(char *dst, const char *src, size_t bytes) {
#if defined(__x86_64__)
    if ((reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
        const size_t lines = bytes / 64;
        for (size_t i = 0; i < lines; i++, dst += 64, src += 64) {
            const __m128i a = _mm_loadu_si128(reinterpret_cast<const __m128i *>(src)), b = _mm_loadu_si128(reinterpret_cast<const __m128i *>(src + 16));
            const __m128i c = _mm_loadu_si128(reinterpret_cast<const __m128i *>(src + 32)), d = _mm_loadu_si128(reinterpret_cast<const __m128i *>(src + 48));
            _mm_stream_si128(reinterpret_cast<__m128i *>(dst), a);
            _mm_stream_si128(reinterpret_cast<__m128i *>(dst + 16), b);
            _mm_stream_si128(reinterpret_cast<__m128i *>(dst + 32), c);
            _mm_stream_si128(reinterpret_cast<__m128i *>(dst + 48), d);
        }
        _mm_sfence();
        bytes -= 64 * lines;
    }
#endif
    memcpy(dst, src, bytes);
}

// ---- pinned buffers ------------------------------------------------------------------------------------------------------
void HostStage::create() {
    auto event = [](hipEvent_t &e) { IOS_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming)); };
    for (int h = 0; h < kParts; h++) {
        IOS_HIP(hipHostMalloc(reinterpret_cast<void **>(&part_[h]), kPart, hipHostMallocDefault));
        event(drained_[h]);
    }
    for (hipEvent_t &e : chunk_events_) event(e);
    event(order_);
    event(sent_);
    event(inputs_.drained);
    event(weights_.drained);
    IOS_HIP(hipHostMalloc(reinterpret_cast<void **>(&result_), kResult, hipHostMallocMapped | hipHostMallocCoherent));
    constexpr size_t kWords = (1 + kResult / kChunk) * sizeof(unsigned);
    IOS_HIP(hipHostMalloc(reinterpret_cast<void **>(&words_), kWords, hipHostMallocMapped | hipHostMallocCoherent));
    memset(words_, 0, kWords);
    IOS_HIP(hipMalloc(reinterpret_cast<void **>(&tickets_), kWords));
    IOS_HIP(hipMemset(tickets_, 0, kWords));
}

char *HostStage::acquire() {
    turn_ = (turn_ + 1) % kParts;
    if (used_[turn_]) {
        used_[turn_] = false;
        IOS_HIP(hipEventSynchronize(drained_[turn_]));
    }
    return part_[turn_];
}

char *HostStage::Batch::take(size_t need) {
    if (used) {
        used = false;
        IOS_HIP(hipEventSynchronize(drained));
    }
    if (need > bytes) {
        if (memory != nullptr) IOS_HIP(hipHostFree(memory));
        memory = nullptr;
        bytes = 0;
        const size_t want = (need + (size_t(16) << 20) - 1) & ~((size_t(16) << 20) - 1);
        IOS_HIP(hipHostMalloc(reinterpret_cast<void **>(&memory), want, hipHostMallocDefault));
        bytes = want;
    }
    return memory;
}

void HostStage::arrived(int chunk, hipStream_t stream) { IOS_HIP(hipStreamWaitEvent(stream, chunk_events_[chunk], 0)); }

void HostStage::upload_chunks(void *dst, const void *src, size_t total, size_t bytes, hipStream_t link, hipStream_t stream) {
    char *memory = inputs_.take(total);
    IOS_HIP(hipEventRecord(order_, stream));
    IOS_HIP(hipStreamWaitEvent(link, order_, 0));
    // one shared-out copy of the whole batch; the calling thread hands a chunk to the link as soon as its pieces are staged
    const int chunks = (int)((total + bytes - 1) / bytes);
    const int per_chunk = (int)((bytes + HostCopier::kPiece - 1) / HostCopier::kPiece);
    std::atomic<int> staged[kMaxChunks] = {};
    auto chunk_bytes = [&](int c) { return std::min(bytes, total - (size_t)c * bytes); };
    int sent = 0;
    hipError_t failed = hipSuccess;
    const std::function<void()> hand_over = [&]() {
        while (sent < chunks && staged[sent].load(std::memory_order_acquire) == per_chunk) {
            const size_t at = (size_t)sent * bytes;
            hipError_t status = hipMemcpyAsync(static_cast<char *>(dst) + at, memory + at, chunk_bytes(sent), hipMemcpyHostToDevice, link);
            if (status == hipSuccess) status = hipEventRecord(chunk_events_[sent], link);
            if (failed == hipSuccess) failed = status;
            sent++;
        }
    };
    HostCopier::get().parallel(chunks * per_chunk, [&](int piece) {
        const int c = piece / per_chunk;
        const size_t at = (size_t)(piece - c * per_chunk) * HostCopier::kPiece, limit = chunk_bytes(c), from = (size_t)c * bytes + at;
        if (at < limit) copy_past_caches(memory + from, static_cast<const char *>(src) + from, std::min(HostCopier::kPiece, limit - at));
        staged[c].fetch_add(1, std::memory_order_release);
    }, &hand_over);
    IOS_HIP(failed);
    IOS_HIP(hipEventRecord(inputs_.drained, link));
    inputs_.used = true;
}

void HostStage::upload_pieces(char *dst, const std::vector<Piece> &all, hipStream_t link, hipStream_t stream, const std::function<void(size_t)> &step) {
    IOS_HIP(hipEventRecord(order_, stream));   // queued passes read what they were queued with
    IOS_HIP(hipStreamWaitEvent(link, order_, 0));
    for (size_t begin = 0; begin < all.size();) {
        // a round: what fits the staging buffer
        size_t end = begin + 1;
        while (end < all.size() && all[end].to + all[end].bytes - all[begin].to <= kBatch) end++;
        const size_t base = all[begin].to, span = all[end - 1].to + all[end - 1].bytes - base;
        char *memory = weights_.take(span);
        // work is handed out in runs of about kPiece bytes; every run is followed by a look at what can be sent
        std::vector<size_t> cuts{begin};
        size_t load = 0;
        for (size_t i = begin; i < end; i++) {
            load += all[i].bytes;
            if (load >= HostCopier::kPiece || i + 1 == end) {
                cuts.push_back(i + 1);
                load = 0;
            }
        }
        const int runs = (int)cuts.size() - 1;
        std::vector<std::atomic<char>> staged(runs);
        for (auto &flag : staged) flag.store(0, std::memory_order_relaxed);
        int ready = 0;
        size_t sent = begin;   // first piece that is not on the link yet
        hipError_t failed = hipSuccess;
        const std::function<void()> hand_over = [&]() {
            while (ready < runs && staged[ready].load(std::memory_order_acquire) != 0) ready++;
            const size_t limit = cuts[ready];
            if (failed != hipSuccess || limit == sent) return;
            const size_t from = all[sent].to, to = all[limit - 1].to + all[limit - 1].bytes;
            if (to - from < kPart && ready < runs) return;
            // pieces with a real gap between them (something else lives there) travel apart
            for (size_t first = sent; first < limit && failed == hipSuccess;) {
                size_t last = first;
                while (last + 1 < limit && all[last + 1].to - (all[last].to + all[last].bytes) < 256) last++;
                failed = hipMemcpyAsync(dst + all[first].to, memory + (all[first].to - base), all[last].to + all[last].bytes - all[first].to,
                                        hipMemcpyHostToDevice, link);
                first = last + 1;
            }
            if (failed == hipSuccess) failed = hipEventRecord(sent_, link);
            if (failed == hipSuccess) failed = hipStreamWaitEvent(stream, sent_, 0);
            sent = limit;
            if (failed == hipSuccess) step(limit);
        };
        HostCopier::get().parallel(runs, [&](int run) {
            for (size_t i = cuts[run]; i < cuts[run + 1]; i++) copy_past_caches(memory + (all[i].to - base), all[i].src, all[i].bytes);
            staged[run].store(1, std::memory_order_release);
        }, &hand_over);
        IOS_HIP(failed);
        IOS_HIP(hipEventRecord(weights_.drained, link));
        weights_.used = true;
        begin = end;
    }
}

// Bound by the link; a kernel that reads host memory reaches its rate with 256 blocks, like the copy engine, and follows and
// precedes the kernels of its stream without the hand-over between engines (600 KB: 25 us less per pass).
__global__ __launch_bounds__(256) void pull_kernel(float *dst, const float *src, unsigned words) {
    const unsigned thread = blockIdx.x * blockDim.x + threadIdx.x, threads = gridDim.x * blockDim.x, quads = words >> 2;
    const float4 *from = reinterpret_cast<const float4 *>(src);
    float4 *to = reinterpret_cast<float4 *>(dst);
    for (unsigned i = thread; i < quads; i += threads) to[i] = from[i];
    for (unsigned i = 4 * quads + thread; i < words; i += threads) dst[i] = src[i];
}

void HostStage::upload(void *dst, const void *src, size_t bytes, hipStream_t stream) {
    if (bytes > kPull || bytes % sizeof(float) != 0) {
        for (size_t at = 0; at < bytes; at += kPart) {
            const size_t n = std::min(kPart, bytes - at);
            char *buffer = acquire();
            HostCopier::get().copy(buffer, static_cast<const char *>(src) + at, n);
            IOS_HIP(hipMemcpyAsync(static_cast<char *>(dst) + at, buffer, n, hipMemcpyHostToDevice, stream));
            IOS_HIP(hipEventRecord(drained_[turn_], stream));
            used_[turn_] = true;
        }
        return;
    }
    // steps of a size that lets the link start before everything is staged
    char *buffer = acquire();
    const size_t step = bytes > (size_t(256) << 10) ? std::max(size_t(128) << 10, (bytes / 4 + 255) & ~size_t(255)) : bytes;
    auto pull = [&](size_t at, size_t n) {
        const unsigned words = (unsigned)(n / sizeof(float));
        hipLaunchKernelGGL(pull_kernel, dim3(std::min(256u, words / 1024 + 1)), dim3(256), 0, stream,
                           reinterpret_cast<float *>(static_cast<char *>(dst) + at), reinterpret_cast<const float *>(buffer + at), words);
    };
    const int steps = (int)((bytes + step - 1) / step);
    auto stage = [&](int s) {
        const size_t at = (size_t)s * step;
        memcpy(buffer + at, static_cast<const char *>(src) + at, std::min(step, bytes - at));
    };
    if (bytes < HostCopier::kParallelBytes) {
        for (int s = 0; s < steps; s++) {
            stage(s);
            pull((size_t)s * step, std::min(step, bytes - (size_t)s * step));
        }
    } else {
        constexpr size_t kSlice = size_t(128) << 10;
        const int slices = (int)((bytes + kSlice - 1) / kSlice);
        std::atomic<char> staged[kPart / kSlice] = {};
        int ready = 0;
        size_t sent = 0;
        const std::function<void()> hand_over = [&]() {
            while (ready < slices && staged[ready].load(std::memory_order_acquire) != 0) ready++;
            const size_t limit = std::min(bytes, (size_t)ready * kSlice);
            if (limit == sent || (limit - sent < step && limit < bytes)) return;
            pull(sent, limit - sent);
            sent = limit;
        };
        HostCopier::get().parallel(slices, [&](int i) {
            const size_t at = (size_t)i * kSlice;
            memcpy(buffer + at, static_cast<const char *>(src) + at, std::min(kSlice, bytes - at));
            staged[i].store(1, std::memory_order_release);
        }, &hand_over);
    }
    IOS_HIP(hipGetLastError());
    IOS_HIP(hipEventRecord(drained_[turn_], stream));
    used_[turn_] = true;
}

void HostStage::download(void *dst, const void *src, size_t bytes, hipStream_t stream) {
    // one part travels while the one before it is copied to the caller; small transfers take one step
    struct Part {
        size_t at, n;
        int part;
    };
    Part last{0, 0, 0};
    const size_t part = bytes > (kPart >> 2) ? kPart >> 2 : kPart;
    size_t at = 0;
    while (at < bytes || last.n > 0) {
        Part now{0, 0, 0};
        if (at < bytes) {
            now.at = at;
            now.n = std::min(part, bytes - at);
            char *buffer = acquire();
            now.part = turn_;
            IOS_HIP(hipMemcpyAsync(buffer, static_cast<const char *>(src) + at, now.n, hipMemcpyDeviceToHost, stream));
            IOS_HIP(hipEventRecord(drained_[turn_], stream));
            at += now.n;
        }
        if (last.n > 0) {
            IOS_HIP(hipEventSynchronize(drained_[last.part]));
            HostCopier::get().copy(static_cast<char *>(dst) + last.at, part_[last.part], last.n);
        }
        last = now;
    }
}

// ---- end of a pass -------------------------------------------------------------------------------------------------------
// Bound by the link (57 GB/s to host memory; 2.5 MB in 44 us, and the caller's copy, 33 us, beside it instead of behind it).
// Four groups of 16 blocks take the chunks in turn: enough stores in flight for the link's rate while a group waits for the
// acknowledgement of its chunk, and the chunks still complete nearly in order (eight groups: 52 instead of 39 us for 1.7 MB).
constexpr int kGroups = 4, kGroupBlocks = 16;
__global__ __launch_bounds__(256) void signal_kernel(float *dst, const float *src, unsigned batch, unsigned image, long long bstride, unsigned chunk,
                                                     unsigned *tickets, unsigned *words, unsigned pass) {
    if (blockIdx.x == 0 && threadIdx.x == 0) __hip_atomic_store(words, pass, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (src == nullptr) return;
    const unsigned total = batch * image;
    const unsigned group_blocks = gridDim.x < kGroupBlocks ? gridDim.x : kGroupBlocks;   // (one block for a single small chunk)
    const unsigned groups = gridDim.x / group_blocks, group = blockIdx.x / group_blocks;
    const unsigned thread = (blockIdx.x - group * group_blocks) * blockDim.x + threadIdx.x, threads = group_blocks * blockDim.x;
    const bool dense = bstride == (long long)image;
    unsigned c = group;
    for (unsigned begin = c * chunk; begin < total; begin += groups * chunk, c += groups) {
        const unsigned end = begin + chunk < total ? begin + chunk : total;
        // stores at system scope go to host memory by themselves: the fence that would send plain ones there writes back the whole
        // L2, block after block (1.7 MB to the caller: 54 instead of 39 us)
        if (dense) {
            const unsigned pairs = (end - begin) >> 1;
            const unsigned long long *from = reinterpret_cast<const unsigned long long *>(src + begin);
            unsigned long long *to = reinterpret_cast<unsigned long long *>(dst + begin);
            for (unsigned i = thread; i < pairs; i += threads) __hip_atomic_store(to + i, from[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            if ((end - begin) & 1u && thread == 0) __hip_atomic_store(dst + end - 1, src[end - 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        } else {
            for (unsigned i = begin + thread; i < end; i += threads) {
                const unsigned b = i / image;
                __hip_atomic_store(dst + i, src[(long long)b * bstride + (i - b * image)], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            }
        }
        // a block's stores are acknowledged before its ticket is drawn; the chunk's last ticket announces it
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x != 0) continue;
        if (group_blocks > 1) {
            if (__hip_atomic_fetch_add(tickets + c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != group_blocks - 1) continue;
            __hip_atomic_store(tickets + c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __hip_atomic_store(words + 1 + c, pass, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

void HostStage::signal(const Result &result, hipStream_t stream) {
    const size_t bytes = result.src != nullptr ? sizeof(float) * (size_t)result.batch * (size_t)result.image : 0;
    if (bytes > kResult) throw std::runtime_error("internal: result larger than its staging buffer");
    pass_++;
    if (bytes > kAlone) HostCopier::get().rouse();
    const int blocks = bytes <= (size_t(16) << 10) ? 1 : bytes <= kChunk ? kGroupBlocks : kGroups * kGroupBlocks;
    hipLaunchKernelGGL(signal_kernel, dim3(blocks), dim3(256), 0, stream, result_, result.src, (unsigned)result.batch, (unsigned)result.image,
                       result.bstride, (unsigned)(kChunk / sizeof(float)), tickets_, words_, pass_);
    IOS_HIP(hipGetLastError());
}

hipError_t HostStage::watch(int word, hipStream_t stream) {
    using clock = std::chrono::steady_clock;
    // the stream itself is asked every now and then: a failed pass never raises the word
    auto next = clock::now() + std::chrono::microseconds(500);
    for (unsigned spins = 0;; spins++) {
        if (__atomic_load_n(words_ + word, __ATOMIC_ACQUIRE) == pass_) return hipSuccess;
        pause();
        if ((spins & 63) != 63 || clock::now() < next) continue;
        const hipError_t status = hipStreamQuery(stream);
        if (status != hipErrorNotReady) return status;
        next = clock::now() + std::chrono::microseconds(500);
    }
}

void HostStage::wait(hipStream_t stream) { IOS_HIP(watch(0, stream)); }

void HostStage::fetch(void *dst, size_t bytes, hipStream_t stream) {
    // memory that a device has just written is read at 25-30 GB/s by one thread: several threads, each waiting for its chunk
    const int chunks = (int)((bytes + kChunk - 1) / kChunk);
    std::atomic<int> failed{hipSuccess};
    const auto body = [&](int c) {
        const hipError_t status = watch(1 + c, stream);
        if (status != hipSuccess) {
            failed.store(status);
            return;
        }
        const size_t at = (size_t)c * kChunk;
        memcpy(static_cast<char *>(dst) + at, reinterpret_cast<const char *>(result_) + at, std::min(kChunk, bytes - at));
    };
    if (bytes <= kAlone) {
        for (int c = 0; c < chunks; c++) body(c);
    } else {
        HostCopier::get().parallel(chunks, body);
    }
    IOS_HIP((hipError_t)failed.load());
}

}  // namespace ios
