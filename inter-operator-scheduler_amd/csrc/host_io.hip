#include "host_io.h"

#include <algorithm>
#include <chrono>
#include <cstring>
#include <stdexcept>

#if defined(__x86_64__)
#include <immintrin.h>
#endif

#include "runtime.h"

namespace ios {

// Fills a buffer that only the link will read and that is larger than the caches: stores past the caches save reading every
// line of the buffer first (a third of the copy's memory traffic).
#if defined(__x86_64__)
__attribute__((target("avx512f"))) static size_t stream_lines_512(char *dst, const char *src, size_t bytes) {
    const size_t whole = bytes & ~size_t(255);
    for (size_t i = 0; i < whole; i += 256) {
        const __m512i a = _mm512_loadu_si512(src + i), b = _mm512_loadu_si512(src + i + 64);
        const __m512i c = _mm512_loadu_si512(src + i + 128), d = _mm512_loadu_si512(src + i + 192);
        _mm512_stream_si512(reinterpret_cast<__m512i *>(dst + i), a);
        _mm512_stream_si512(reinterpret_cast<__m512i *>(dst + i + 64), b);
        _mm512_stream_si512(reinterpret_cast<__m512i *>(dst + i + 128), c);
        _mm512_stream_si512(reinterpret_cast<__m512i *>(dst + i + 192), d);
    }
    _mm_sfence();
    return whole;
}
static size_t stream_lines_128(char *dst, const char *src, size_t bytes) {
    const size_t whole = bytes & ~size_t(63);
    for (size_t i = 0; i < whole; i += 16)
        _mm_stream_si128(reinterpret_cast<__m128i *>(dst + i), _mm_loadu_si128(reinterpret_cast<const __m128i *>(src + i)));
    _mm_sfence();
    return whole;
}
#endif

static void copy_past_caches(char *dst, const char *src, size_t bytes) {
    size_t done = 0;
#if defined(__x86_64__)
    static const bool wide = __builtin_cpu_supports("avx512f");
    if ((reinterpret_cast<uintptr_t>(dst) & 63) == 0) done = wide ? stream_lines_512(dst, src, bytes) : stream_lines_128(dst, src, bytes);
#endif
    memcpy(dst + done, src + done, bytes - done);
}

// A transfer that fails midway may have queued steps on `stream` that still read the staging buffers: they end before the buffers
// are used again.
namespace {
struct SettleOnFailure {
    hipStream_t stream;
    bool armed = true;
    ~SettleOnFailure() {
        if (armed) (void)hipStreamSynchronize(stream);
    }
};
}  // namespace

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

void HostStage::give_back() noexcept {
    for (Batch *b : {&inputs_, &weights_}) {
        if (b->bytes <= kIdle) continue;
        (void)hipHostFree(b->memory);
        b->memory = nullptr;
        b->bytes = 0;
        b->used = false;
    }
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

// Kernels read the staging buffer at the link's rate, like the copy engine, turn the images into the layout of views on the
// way, and follow and precede the kernels of their stream without the hand-over between engines (600 KB: 25 us less per pass).
void HostStage::upload_images(const TensorView &dst, int batch, const float *src, hipStream_t stream) {
    SettleOnFailure settle{stream};
    const size_t pixels = (size_t)dst.H * dst.W, image = pixels * dst.C;   // floats
    const int group = (int)std::max<size_t>(1, std::min<size_t>((size_t)batch, kBatch / (image * sizeof(float))));
    struct Step {
        TensorView part;
        const float *from;
        int images, pieces;
        long long plane;
    };
    struct Copy {
        size_t at, floats;   // in the group
        int step;
    };
    std::vector<Step> steps;
    std::vector<Copy> copies;
    for (int first = 0; first < batch; first += group) {
        const int images = std::min(group, batch - first);
        const size_t floats = (size_t)images * image, bytes = floats * sizeof(float);
        const bool ring = bytes <= kPart;
        float *memory = reinterpret_cast<float *>(ring ? acquire() : inputs_.take(bytes));
        const float *host = src + (size_t)first * image;
        TensorView view = dst;
        view.ptr += (size_t)first * pixels * dst.pstride;
        // Steps, so that the link starts before everything is staged (a third at a time and 768 KB at least: a step of 150 KB takes
        // 5 us and the launch of the next one another 5): whole images, or bands of pixels (few channels) or of channels of a
        // single one.  Every step is copied in pieces.
        steps.clear();
        copies.clear();
        const size_t step_floats = std::max(size_t(192) << 10, std::min((floats + 2) / 3, size_t(512) << 10));
        const size_t piece_floats = std::max(size_t(8) << 10, std::min(floats / 16, HostCopier::kPiece / sizeof(float)));
        auto add_copy = [&](size_t at, size_t n) {
            for (size_t p = 0; p < n; p += piece_floats) {
                copies.push_back({at + p, std::min(piece_floats, n - p), (int)steps.size() - 1});
                steps.back().pieces++;
            }
        };
        if (images > 1) {
            const int per_step = (int)std::max<size_t>(1, step_floats / image);
            for (int i = 0; i < images; i += per_step) {
                Step s{view, memory + i * image, std::min(per_step, images - i), 0, 0};
                s.part.ptr += (size_t)i * pixels * dst.pstride;
                steps.push_back(s);
                add_copy(i * image, s.images * image);
            }
        } else if (dst.C <= 4) {
            const size_t band = (step_floats / dst.C + 63) & ~size_t(63);
            for (size_t p = 0; p < pixels; p += band) {
                const size_t n = std::min(band, pixels - p);
                Step s{view, memory + p, 1, 0, (long long)pixels};
                s.part.ptr += p * dst.pstride;
                s.part.H = 1;
                s.part.W = (int)n;
                steps.push_back(s);
                for (int c = 0; c < dst.C; c++) add_copy(c * pixels + p, n);
            }
        } else {
            const int band = (int)((step_floats / pixels + 32) & ~size_t(31));
            for (int c = 0; c < dst.C; c += band) {
                Step s{view, memory + c * pixels, 1, 0, 0};
                s.part.ptr += c;
                s.part.C = std::min(band, dst.C - c);
                steps.push_back(s);
                add_copy(c * pixels, s.part.C * pixels);
            }
        }
        auto copy = [&](const Copy &c) {
            char *to = reinterpret_cast<char *>(memory + c.at);
            const char *from = reinterpret_cast<const char *>(host + c.at);
            if (ring) memcpy(to, from, c.floats * sizeof(float));
            else copy_past_caches(to, from, c.floats * sizeof(float));
        };
        if (bytes <= HostCopier::kAloneBytes) {
            size_t next = 0;
            for (size_t s = 0; s < steps.size(); s++) {
                for (; next < copies.size() && copies[next].step == (int)s; next++) copy(copies[next]);
                launch_to_view(steps[s].from, steps[s].part, steps[s].images, stream, steps[s].plane);
            }
        } else {
            // one shared-out copy; the calling thread hands a step to the link as soon as its pieces are staged
            std::vector<std::atomic<int>> staged(steps.size());
            for (auto &count : staged) count.store(0, std::memory_order_relaxed);
            size_t sent = 0;
            const std::function<void()> hand_over = [&]() {
                for (; sent < steps.size() && staged[sent].load(std::memory_order_acquire) == steps[sent].pieces; sent++)
                    launch_to_view(steps[sent].from, steps[sent].part, steps[sent].images, stream, steps[sent].plane);
            };
            HostCopier::get().parallel((int)copies.size(), bytes >= HostCopier::kLargeBytes, [&](int i) {
                copy(copies[i]);
                staged[copies[i].step].fetch_add(1, std::memory_order_release);
            }, &hand_over);
        }
        IOS_HIP(hipGetLastError());
        IOS_HIP(hipEventRecord(ring ? drained_[turn_] : inputs_.drained, stream));
        if (ring) used_[turn_] = true;
        else inputs_.used = true;
    }
    settle.armed = false;
}

void HostStage::upload_chunks(void *dst, const void *src, const std::vector<size_t> &ends, hipStream_t link, hipStream_t stream) {
    SettleOnFailure settle{link};
    const int chunks = (int)ends.size();
    if (chunks < 1 || chunks > kMaxChunks) throw std::runtime_error("internal: a batch arrives in too many chunks");
    char *memory = inputs_.take(ends.back());
    IOS_HIP(hipEventRecord(order_, stream));
    IOS_HIP(hipStreamWaitEvent(link, order_, 0));
    // one shared-out copy of the whole batch; the calling thread hands a chunk to the link as soon as its pieces are staged
    auto begin_of = [&](int c) { return c == 0 ? 0 : ends[c - 1]; };
    int first_piece[kMaxChunks + 1] = {};
    for (int c = 0; c < chunks; c++) first_piece[c + 1] = first_piece[c] + (int)((ends[c] - begin_of(c) + HostCopier::kPiece - 1) / HostCopier::kPiece);
    std::atomic<int> staged[kMaxChunks] = {};
    int sent = 0;
    hipError_t failed = hipSuccess;
    const std::function<void()> hand_over = [&]() {
        while (sent < chunks && staged[sent].load(std::memory_order_acquire) == first_piece[sent + 1] - first_piece[sent]) {
            const size_t at = begin_of(sent);
            hipError_t status = hipMemcpyAsync(static_cast<char *>(dst) + at, memory + at, ends[sent] - at, hipMemcpyHostToDevice, link);
            if (status == hipSuccess) status = hipEventRecord(chunk_events_[sent], link);
            if (failed == hipSuccess) failed = status;
            sent++;
        }
    };
    HostCopier::get().parallel(first_piece[chunks], true, [&](int piece) {
        int c = 0;
        while (piece >= first_piece[c + 1]) c++;
        const size_t from = begin_of(c) + (size_t)(piece - first_piece[c]) * HostCopier::kPiece;
        copy_past_caches(memory + from, static_cast<const char *>(src) + from, std::min(HostCopier::kPiece, ends[c] - from));
        staged[c].fetch_add(1, std::memory_order_release);
    }, &hand_over);
    IOS_HIP(failed);
    IOS_HIP(hipEventRecord(inputs_.drained, link));
    inputs_.used = true;
    settle.armed = false;
}

void HostStage::upload_pieces(char *dst, const std::vector<Piece> &all, hipStream_t link, hipStream_t stream, const std::function<void(size_t)> &step) {
    SettleOnFailure settle{link};
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
        HostCopier::get().parallel(runs, span >= HostCopier::kLargeBytes, [&](int run) {
            for (size_t i = cuts[run]; i < cuts[run + 1]; i++) copy_past_caches(memory + (all[i].to - base), all[i].src, all[i].bytes);
            staged[run].store(1, std::memory_order_release);
        }, &hand_over);
        IOS_HIP(failed);
        IOS_HIP(hipEventRecord(weights_.drained, link));
        weights_.used = true;
        begin = end;
    }
    settle.armed = false;
}

void HostStage::upload(void *dst, const void *src, size_t bytes, hipStream_t stream) {
    SettleOnFailure settle{stream};
    for (size_t at = 0; at < bytes; at += kPart) {
        const size_t n = std::min(kPart, bytes - at);
        char *buffer = acquire();
        HostCopier::get().copy(buffer, static_cast<const char *>(src) + at, n);
        IOS_HIP(hipMemcpyAsync(static_cast<char *>(dst) + at, buffer, n, hipMemcpyHostToDevice, stream));
        IOS_HIP(hipEventRecord(drained_[turn_], stream));
        used_[turn_] = true;
    }
    settle.armed = false;
}

// Elements [first, first + count) of a view in the host's layout, to host memory (count <= 2^20).  Bound by the link: a part of
// 1 MB is 18 us of it, the gather reads the caches.  A copy engine in place of these stores needs the tensor turned in device
// memory first, as much of it as the tensor itself.
__global__ __launch_bounds__(256) void gather_kernel(float *__restrict__ dst, const float *__restrict__ src, long long first, unsigned count, long long image,
                                                     long long plane, int pstride) {
    for (unsigned i = blockIdx.x * 256u + threadIdx.x; i < count; i += gridDim.x * 256u) {
        const long long e = first + i, b = e / image, rest = e - b * image, c = rest / plane;
        dst[i] = src[(b * plane + rest - c * plane) * pstride + c];
    }
}

void HostStage::download(float *dst, const TensorView &src, int batch, hipStream_t stream) {
    SettleOnFailure settle{stream};
    // one part is gathered while the one before it is copied to the caller; small transfers take one step
    struct Part {
        size_t at, n;   // floats
        int part;
    };
    const long long plane = (long long)src.H * src.W, image = plane * src.C;
    const size_t floats = (size_t)batch * (size_t)image;
    Part last{0, 0, 0};
    const size_t part = floats > (kPart >> 4) ? kPart >> 4 : kPart >> 2;
    size_t at = 0;
    while (at < floats || last.n > 0) {
        Part now{0, 0, 0};
        if (at < floats) {
            now.at = at;
            now.n = std::min(part, floats - at);
            float *buffer = reinterpret_cast<float *>(acquire());
            now.part = turn_;
            hipLaunchKernelGGL(gather_kernel, dim3((unsigned)std::min<size_t>((now.n + 255) / 256, 256)), dim3(256), 0, stream, buffer, src.ptr, (long long)now.at,
                               (unsigned)now.n, image, plane, src.pstride);
            IOS_HIP(hipGetLastError());
            IOS_HIP(hipEventRecord(drained_[turn_], stream));
            at += now.n;
        }
        if (last.n > 0) {
            IOS_HIP(hipEventSynchronize(drained_[last.part]));
            HostCopier::get().copy(dst + last.at, part_[last.part], last.n * sizeof(float));
        }
        last = now;
    }
    settle.armed = false;
}

// ---- end of a pass -------------------------------------------------------------------------------------------------------
// Bound by the link (57 GB/s to host memory; 2.5 MB in 44 us, and the caller's copy, 33 us, beside it instead of behind it).
// Four groups of 16 blocks take the chunks in turn: enough stores in flight for the link's rate while a group waits for the
// acknowledgement of its chunk, and the chunks still complete nearly in order (eight groups: 52 instead of 39 us for 1.7 MB).
constexpr int kGroups = 4, kGroupBlocks = 16;
struct SignalArgs {
    float *dst;
    const float *src;
    unsigned total, image, plane, chunk;   // floats of the result, of an image, pixels of an image; floats of a chunk
    int pstride;
    unsigned *tickets, *words, pass;
    FastDiv div_image, div_plane;
};
__global__ __launch_bounds__(256) void signal_kernel(SignalArgs a) {
    if (blockIdx.x == 0 && threadIdx.x == 0) __hip_atomic_store(a.words, a.pass, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (a.src == nullptr) return;
    const unsigned group_blocks = gridDim.x < kGroupBlocks ? gridDim.x : kGroupBlocks;   // (one block for a single small chunk)
    const unsigned groups = gridDim.x / group_blocks, group = blockIdx.x / group_blocks;
    const unsigned thread = (blockIdx.x - group * group_blocks) * blockDim.x + threadIdx.x, threads = group_blocks * blockDim.x;
    // element i of the host's layout (gathered through the caches: the link is the bound)
    auto element = [&](unsigned i) -> float {
        const unsigned b = fast_div(i, a.div_image), rest = i - b * a.image;
        const unsigned c = fast_div(rest, a.div_plane), r = rest - c * a.plane;
        return a.src[(long long)(b * a.plane + r) * a.pstride + c];
    };
    unsigned c = group;
    for (unsigned begin = c * a.chunk; begin < a.total; begin += groups * a.chunk, c += groups) {
        const unsigned end = begin + a.chunk < a.total ? begin + a.chunk : a.total;
        // stores at system scope go to host memory by themselves: the fence that would send plain ones there writes back the whole
        // L2, block after block (1.7 MB to the caller: 54 instead of 39 us)
        const unsigned pairs = (end - begin) >> 1;
        unsigned long long *to = reinterpret_cast<unsigned long long *>(a.dst + begin);
        for (unsigned i = thread; i < pairs; i += threads) {
            const unsigned low = __float_as_uint(element(begin + 2 * i)), high = __float_as_uint(element(begin + 2 * i + 1));
            __hip_atomic_store(to + i, (unsigned long long)high << 32 | low, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        if ((end - begin) & 1u && thread == 0) __hip_atomic_store(a.dst + end - 1, element(end - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        // a block's stores are acknowledged before its ticket is drawn; the chunk's last ticket announces it
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x != 0) continue;
        if (group_blocks > 1) {
            if (__hip_atomic_fetch_add(a.tickets + c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != group_blocks - 1) continue;
            __hip_atomic_store(a.tickets + c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __hip_atomic_store(a.words + 1 + c, a.pass, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

unsigned HostStage::signal(const Result &result, hipStream_t stream) {
    const TensorView &v = result.view;
    SignalArgs a{};
    a.dst = result_;
    a.src = v.ptr;
    a.plane = v.ptr != nullptr ? (unsigned)(v.H * v.W) : 1;
    a.image = v.ptr != nullptr ? a.plane * (unsigned)v.C : 1;
    a.total = v.ptr != nullptr ? (unsigned)result.batch * a.image : 0;
    a.chunk = (unsigned)(kChunk / sizeof(float));
    a.pstride = v.pstride;
    a.tickets = tickets_;
    a.words = words_;
    a.pass = ++pass_;
    a.div_image = make_fast_div(a.image);
    a.div_plane = make_fast_div(a.plane);
    const size_t bytes = sizeof(float) * (size_t)a.total;
    if (bytes > kResult) throw std::runtime_error("internal: result larger than its staging buffer");
    if (bytes > kAlone) HostCopier::get().rouse();
    const int blocks = bytes <= (size_t(16) << 10) ? 1 : bytes <= kChunk ? kGroupBlocks : kGroups * kGroupBlocks;
    hipLaunchKernelGGL(signal_kernel, dim3(blocks), dim3(256), 0, stream, a);
    IOS_HIP(hipGetLastError());
    return a.pass;
}

hipError_t HostStage::watch(int word, unsigned pass, hipStream_t stream) {
    using clock = std::chrono::steady_clock;
    // the stream itself is asked every now and then: a failed pass never raises the word
    auto next = clock::now() + std::chrono::microseconds(500);
    for (unsigned spins = 0;; spins++) {
        if (__atomic_load_n(words_ + word, __ATOMIC_ACQUIRE) == pass) return hipSuccess;
        spin_pause();
        if ((spins & 63) != 63 || clock::now() < next) continue;
        const hipError_t status = hipStreamQuery(stream);
        if (status != hipErrorNotReady) return status;
        next = clock::now() + std::chrono::microseconds(500);
    }
}

void HostStage::wait(unsigned pass, hipStream_t stream) { IOS_HIP(watch(0, pass, stream)); }

void HostStage::fetch(void *dst, size_t bytes, unsigned pass, hipStream_t stream) {
    // memory that a device has just written is read at 25-30 GB/s by one thread: several threads, each waiting for its chunk
    const int chunks = (int)((bytes + kChunk - 1) / kChunk);
    std::atomic<int> failed{hipSuccess};
    const auto body = [&](int c) {
        const hipError_t status = watch(1 + c, pass, stream);
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
        HostCopier::get().parallel(chunks, false, body);
    }
    IOS_HIP((hipError_t)failed.load());
}

}  // namespace ios
