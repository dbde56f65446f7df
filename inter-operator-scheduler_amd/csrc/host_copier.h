// Copies of host memory, shared out over several threads.  Plain C++: nothing here touches the device.
#pragma once

#include <atomic>
#include <cstddef>
#include <exception>
#include <functional>
#include <mutex>

namespace ios {

inline void spin_pause() {
#if defined(__x86_64__)
    __builtin_ia32_pause();
#endif
}

// Shares out copies of host memory over several threads.  They are started on the first large copy, sleep between copies (on
// futexes) and stay with the process (the pool is never destroyed: a sleeping thread must not touch it while the process
// unloads).  Waking a thread takes 20-40 us, longer than a 1 MB copy: three of them, the near ones, stay awake for half a
// millisecond behind a copy, so that a caller who serves one request after the other finds them; the far ones join large copies
// only.
class HostCopier {
public:
    static HostCopier &get();
    // `pieces` bodies, taken in order by the calling thread and the workers; `idle`, if given, is called by the calling thread
    // between its pieces and until all are done; `large`: the far workers take part.  Where one of them throws, no further piece is
    // begun, the exception passes on once no thread is inside `body` any more, and the next copy starts afresh.
    void parallel(int pieces, bool large, const std::function<void(int)> &body, const std::function<void()> *idle = nullptr);
    void copy(void *dst, const void *src, size_t bytes);
    void rouse();   // a copy is to come within half a millisecond: the near workers wake up for it
    static constexpr size_t kAloneBytes = size_t(192) << 10;   // one thread's copy (8 us) up to here
    static constexpr size_t kLargeBytes = size_t(8) << 20;
    static constexpr size_t kPiece = size_t(512) << 10;

private:
    HostCopier() = default;
    void start();
    void worker(bool near);
    static constexpr int kNear = 3;
    bool started_ = false;
    const std::function<void(int)> *body_ = nullptr;
    int pieces_ = 0;
    std::atomic<unsigned> generation_{0};                        // number of the copy
    std::atomic<unsigned> open_{0};                              // generation of the copy that workers may join (0: none)
    std::atomic<unsigned> near_calls_{0}, far_calls_{0};         // futex words
    std::atomic<int> near_asleep_{0}, far_asleep_{0};
    std::atomic<int> next_{0}, busy_{0};
    std::mutex failure_mutex_;
    std::exception_ptr failure_;                                 // what a worker's piece threw
};

}  // namespace ios
