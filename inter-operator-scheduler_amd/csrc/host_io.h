// Host side of the boundary: moving tensors between a caller's pageable memory and the device, and waiting for a pass.
//
// A copy from or to pageable memory makes the driver pin, stage or bounce the caller's pages inside the call: 2.5 MB leave
// the device in 151 us and 69 MB reach it in 2.56 ms that way, against 52 us and 1.20 ms (57 GB/s, the link's rate) from
// memory that is pinned already.  So every transfer goes through a few pinned buffers that live as long as the device
// context: a few host threads fill one part (8 threads copy 69 MB in 0.31 ms, one in 2.4 ms) while the link drains the others.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <functional>
#include <vector>

namespace ios {

// Shares out copies of host memory over several threads.  They are started on the first large copy, sleep between copies
// (on a futex: waking seven threads through a mutex took longer than their share of an 8 MB copy), and stay with the process
// (the pool is never destroyed: a sleeping thread must not touch it while the process unloads).
class HostCopier {
public:
    static HostCopier &get();
    // `pieces` bodies, taken in order by the calling thread and the workers; `idle`, if given, is called by the calling thread
    // between its pieces and until all are done
    void parallel(int pieces, const std::function<void(int)> &body, const std::function<void()> *idle = nullptr);
    void copy(void *dst, const void *src, size_t bytes);
    // A few workers wake up and wait, awake, for a copy that is to come within a millisecond (waking a sleeping thread takes 20 to
    // 40 us, as long as copying a 1.7 MB result).
    void rouse();
    // below this one thread is faster than waking others (2.5 MB: 33 us with one thread, 4-11 us with workers that are awake)
    static constexpr size_t kParallelBytes = size_t(3) << 19;
    static constexpr size_t kPiece = size_t(256) << 10;

private:
    HostCopier() = default;
    void start();
    void worker();
    bool started_ = false;
    const std::function<void(int)> *body_ = nullptr;
    int pieces_ = 0;
    std::atomic<unsigned> generation_{0};   // number of the copy
    std::atomic<unsigned> calls_{0};        // the futex word: changes with every copy and every rouse()
    std::atomic<unsigned> open_{0};         // generation of the copy that workers may join (0: none)
    std::atomic<int> next_{0}, busy_{0};
};

class HostStage {
public:
    static constexpr size_t kPart = size_t(4) << 20;      // bytes per staging buffer of the ring, and per step of a large transfer
    static constexpr int kParts = 4;
    static constexpr int kMaxChunks = 8;                  // steps in which a batch arrives
    static constexpr size_t kBatch = size_t(256) << 20;   // largest transfer that is staged as a whole
    static constexpr size_t kPull = kPart;                // largest upload that a kernel reads from host memory
    static constexpr size_t kChunk = size_t(64) << 10;   // bytes of the result that are announced together
    static constexpr size_t kAlone = 3 * kChunk;          // results up to this size are fetched by one thread
    static constexpr size_t kResult = size_t(4) << 20;    // largest result a pass delivers to host memory by itself

    void create();   // with the device context (pinned memory goes with the process: the runtime may be unloaded before static objects are)

    // Copies `bytes` to the device behind what `stream` holds.  Returns when the caller's memory may change again; the
    // last part may still be on its way (in stream order).
    void upload(void *dst, const void *src, size_t bytes, hipStream_t stream);
    // The same for a batch of `total` <= kBatch bytes in chunks of `bytes` bytes each (the last may be shorter), on the stream
    // `link` behind what `stream` holds: chunk c has arrived for a stream that called arrived(c, stream).
    void upload_chunks(void *dst, const void *src, size_t total, size_t bytes, hipStream_t link, hipStream_t stream);
    void arrived(int chunk, hipStream_t stream);
    // Scattered sources that lie next to each other on the device: `pieces` ascending by `to`, an offset from `dst`, without
    // overlap, gaps of less than a cache line's worth of padding that may be overwritten.  `step` is called by the calling thread
    // whenever the bytes up to a limit have been sent, after `stream` was told to wait for them.
    struct Piece {
        size_t to, bytes;
        const char *src;
    };
    void upload_pieces(char *dst, const std::vector<Piece> &pieces, hipStream_t link, hipStream_t stream, const std::function<void(size_t)> &step);
    // Device to host, complete on return.
    void download(void *dst, const void *src, size_t bytes, hipStream_t stream);

    // Waiting for a pass: a last small kernel raises a word in host memory that the caller watches (a kernel and this
    // wait take 5.8 us where hipStreamSynchronize takes 9.5).  Where the result is small or the caller is known to fetch
    // it, the same kernel then writes it to pinned memory, chunk after chunk with a word for each, so that copying a chunk
    // to the caller runs beside the transfer of the ones behind it.
    struct Result {
        const float *src = nullptr;   // null: only the word
        int batch = 0;
        long long image = 0, bstride = 0;   // floats
    };
    void signal(const Result &result, hipStream_t stream);
    void wait(hipStream_t stream);                                  // for the pass behind the last signal()
    void fetch(void *dst, size_t bytes, hipStream_t stream);        // that pass's result

private:
    char *acquire();   // the ring's next buffer, once the link has drained it
    struct Batch {     // a buffer that grows to the transfer it stages, and is kept
        char *memory = nullptr;
        size_t bytes = 0;
        hipEvent_t drained = nullptr;
        bool used = false;
        char *take(size_t need);
    };
    hipError_t watch(int word, hipStream_t stream);
    char *part_[kParts] = {};
    hipEvent_t drained_[kParts] = {};
    bool used_[kParts] = {};
    int turn_ = 0;
    hipEvent_t order_ = nullptr, sent_ = nullptr;
    Batch inputs_, weights_;
    hipEvent_t chunk_events_[kMaxChunks] = {};
    float *result_ = nullptr;
    unsigned *words_ = nullptr;     // host memory: [0] the pass, [1 + c] chunk c of its result, each the number of the pass
    unsigned *tickets_ = nullptr;   // device memory, one per chunk, zero between kernels
    unsigned pass_ = 0;
};

}  // namespace ios
