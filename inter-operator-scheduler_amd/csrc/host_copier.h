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
    // Threads that share a copy, the caller among them; 0: three quarters of the processors this process may use, twelve at most.
    // Threads beyond a lower number sleep.
    void set_threads(int count);
    int threads();
    static constexpr size_t kAloneBytes = size_t(192) << 10;   // one thread's copy (8 us) up to here
    static constexpr size_t kLargeBytes = size_t(8) << 20;
    static constexpr size_t kPiece = size_t(512) << 10;

private:
    HostCopier() = default;
    void start();
    void worker(int index);
    static constexpr int kNear = 3;
    static constexpr int kMost = 12;   // large copies are bound by memory from there on (69 MB that lie in no cache: 530 us with 8 threads, 420 with 12 and with 15)
    int started_ = 1;                                            // threads there are, the caller among them
    std::atomic<int> limit_{0};                                  // threads that take part (0: not chosen yet)
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

// Processors this process may use: those it is bound to, and the share that the control groups above it leave it.
int available_processors();
// Of a control group's limit ("max 100000", "400000 100000": microseconds of processor time in a period): processors, rounded up;
// 0 where there is no limit.
int processors_of_quota(const char *cpu_max);

}  // namespace ios
