#include "host_copier.h"

#include <algorithm>
#include <chrono>
#include <climits>
#include <cstring>
#include <system_error>
#include <thread>

#include <linux/futex.h>
#include <sys/syscall.h>
#include <unistd.h>

namespace ios {

HostCopier &HostCopier::get() {
    static HostCopier *instance = new HostCopier();
    return *instance;
}

static void futex_wait(std::atomic<unsigned> &word, unsigned value) {
    syscall(SYS_futex, reinterpret_cast<unsigned *>(&word), FUTEX_WAIT_PRIVATE, value, nullptr, nullptr, 0);
}
static void futex_wake(std::atomic<unsigned> &word) {
    syscall(SYS_futex, reinterpret_cast<unsigned *>(&word), FUTEX_WAKE_PRIVATE, INT_MAX, nullptr, nullptr, 0);
}

void HostCopier::start() {
    started_ = true;
    // three quarters of the processors, twelve threads at most: large copies are bound by memory from there on (69 MB that lie in no
    // cache: 530 us with 8 threads, 420 with 12 and with 15)
    const int n = std::min(12, std::max(1, (int)std::thread::hardware_concurrency() * 3 / 4));
    try {
        for (int i = 1; i < n; i++) std::thread([this, i]() { worker(i <= kNear); }).detach();
    } catch (const std::system_error &) {   // no more threads to be had: the ones there are do
    }
}

void HostCopier::worker(bool near) {
    using clock = std::chrono::steady_clock;
    std::atomic<unsigned> &calls = near ? near_calls_ : far_calls_;
    std::atomic<int> &asleep = near ? near_asleep_ : far_asleep_;
    unsigned seen = 0;
    for (;;) {
        const unsigned call = calls.load();
        unsigned now = generation_.load();
        if (now == seen && near) {
            const auto until = clock::now() + std::chrono::microseconds(500);
            while ((now = generation_.load()) == seen && clock::now() < until)
                for (int i = 0; i < 32; i++) spin_pause();
        }
        if (now == seen) {
            asleep.fetch_add(1);
            futex_wait(calls, call);
            asleep.fetch_sub(1);
            continue;
        }
        seen = now;
        // either the owner sees this thread in busy_ and waits for it, or this thread sees that the copy is closed
        busy_.fetch_add(1);
        if (open_.load() == now) {
            try {
                for (int i; (i = next_.fetch_add(1)) < pieces_;) (*body_)(i);
            } catch (...) {
                next_.store(pieces_);
                std::lock_guard<std::mutex> lock(failure_mutex_);
                if (!failure_) failure_ = std::current_exception();
            }
        }
        busy_.fetch_sub(1);
    }
}

void HostCopier::rouse() {
    if (!started_) start();
    near_calls_.fetch_add(1);
    if (near_asleep_.load() > 0) futex_wake(near_calls_);
}

void HostCopier::parallel(int pieces, bool large, const std::function<void(int)> &body, const std::function<void()> *idle) {
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
    near_calls_.fetch_add(1);
    if (near_asleep_.load() > 0) futex_wake(near_calls_);
    if (large) {
        far_calls_.fetch_add(1);
        if (far_asleep_.load() > 0) futex_wake(far_calls_);
    }
    std::exception_ptr failure;
    auto guarded = [&](auto &&work) {
        if (failure) return;
        try {
            work();
        } catch (...) {
            failure = std::current_exception();
            next_.store(pieces);
        }
    };
    guarded([&] {
        for (int i; (i = next_.fetch_add(1)) < pieces;) {
            body(i);
            if (idle != nullptr) (*idle)();
        }
    });
    open_.store(0);
    while (busy_.load() != 0) {   // whatever happened: the workers read this call's variables
        if (idle != nullptr) guarded(*idle);
        spin_pause();
    }
    if (failure_) {
        if (!failure) failure = failure_;
        failure_ = nullptr;
    }
    if (failure) std::rethrow_exception(failure);
    if (idle != nullptr) (*idle)();
}

void HostCopier::copy(void *dst, const void *src, size_t bytes) {
    if (bytes <= kAloneBytes) {
        memcpy(dst, src, bytes);
        return;
    }
    const size_t piece = std::min(kPiece, std::max(size_t(32) << 10, bytes / 16));
    parallel((int)((bytes + piece - 1) / piece), bytes >= kLargeBytes, [&](int i) {
        const size_t at = (size_t)i * piece;
        memcpy(static_cast<char *>(dst) + at, static_cast<const char *>(src) + at, std::min(piece, bytes - at));
    });
}

}  // namespace ios
