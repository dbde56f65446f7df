// Host side of the boundary: moving tensors between a caller's pageable memory and the device, and waiting for a pass.
//
// A copy from or to pageable memory makes the driver pin, stage or bounce the caller's pages inside the call: 2.5 MB leave
// the device in 151 us and 69 MB reach it in 2.56 ms that way, against 52 us and 1.20 ms (57 GB/s, the link's rate) from
// memory that is pinned already.  So every transfer goes through a few pinned buffers that live as long as the device
// context: a few host threads fill one part (twelve copy 69 MB that lie in no cache in 0.42 ms, one in 2.4 ms) while the link
// drains the others.
#pragma once

#include <hip/hip_runtime.h>

#include <functional>
#include <vector>

#include "host_copier.h"
#include "plan.h"

namespace ios {

class HostStage {
public:
    static constexpr size_t kPart = size_t(4) << 20;      // bytes per staging buffer of the ring, and per step of a large transfer
    static constexpr int kParts = 4;
    static constexpr int kMaxChunks = 5;                  // steps in which a batch arrives (the copy engine takes 25-35 us from one to the next)
    static constexpr size_t kBatch = kStagedBytes;        // largest transfer that is staged as a whole (or one image)
    static constexpr size_t kIdle = size_t(16) << 20;     // of each growing buffer that stays while there is no session
    static constexpr size_t kChunk = size_t(64) << 10;   // bytes of the result that are announced together
    static constexpr size_t kAlone = 3 * kChunk;          // results up to this size are fetched by one thread
    static constexpr size_t kResult = kDeliveredFloats * sizeof(float);   // largest result a pass delivers to host memory by itself

    // Frees what the growing buffers hold beyond kIdle.  Nothing may be on its way.
    void give_back() noexcept;
    size_t staged_bytes() const { return inputs_.bytes + weights_.bytes; }
    void create();   // with the device context (pinned memory goes with the process: the runtime may be unloaded before static objects are)

    // Copies `bytes` to the device behind what `stream` holds.  Returns when the caller's memory may change again; the
    // last part may still be on its way (in stream order).
    void upload(void *dst, const void *src, size_t bytes, hipStream_t stream);
    // The same for a batch of images in the host's layout, which kernels read from the staging buffer and write as a view.
    void upload_images(const TensorView &dst, int batch, const float *src, hipStream_t stream);
    // A batch of at most kBatch bytes to device memory as it is, in up to kMaxChunks chunks that end at `ends` (bytes), by the
    // copy engine and on the stream `link`, which waits for what `stream` holds: chunk c has arrived for a stream that called
    // arrived(c, stream).  (Kernels that read host memory would share the device with those of `stream`.)
    void upload_chunks(void *dst, const void *src, const std::vector<size_t> &ends, hipStream_t link, hipStream_t stream);
    void arrived(int chunk, hipStream_t stream);
    // Scattered sources that lie next to each other on the device: `pieces` ascending by `to`, an offset from `dst`, without
    // overlap, gaps of less than a cache line's worth of padding that may be overwritten.  `step` is called by the calling thread
    // whenever the bytes up to a limit have been sent, after `stream` was told to wait for them.
    struct Piece {
        size_t to, bytes;
        const char *src;
    };
    void upload_pieces(char *dst, const std::vector<Piece> &pieces, hipStream_t link, hipStream_t stream, const std::function<void(size_t)> &step);
    // A tensor to the caller in the host's layout, complete on return.  Kernels gather it into the staging buffers, so it needs
    // no device memory.
    void download(float *dst, const TensorView &src, int batch, hipStream_t stream);

    // Waiting for a pass: a last small kernel raises a word in host memory that the caller watches (a kernel and this
    // wait take 5.8 us where hipStreamSynchronize takes 9.5).  Where the result is small or the caller is known to fetch
    // it, the same kernel then writes it to pinned memory, chunk after chunk with a word for each, so that copying a chunk
    // to the caller runs beside the transfer of the ones behind it.
    struct Result {
        TensorView view;   // ptr null: only the word
        int batch = 0;
    };
    unsigned signal(const Result &result, hipStream_t stream);      // the number of the pass
    void wait(unsigned pass, hipStream_t stream);
    // The result of a pass that delivered one, until the next pass that does.
    void fetch(void *dst, size_t bytes, unsigned pass, hipStream_t stream);

private:
    char *acquire();   // the ring's next buffer, once the link has drained it
    struct Batch {     // a buffer that grows to the transfer it stages, and is kept while there are sessions
        char *memory = nullptr;
        size_t bytes = 0;
        hipEvent_t drained = nullptr;
        bool used = false;
        char *take(size_t need);
    };
    hipError_t watch(int word, unsigned pass, hipStream_t stream);
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
