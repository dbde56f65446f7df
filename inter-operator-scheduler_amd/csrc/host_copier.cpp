#include "host_copier.h"

#include <algorithm>
#include <chrono>
#include <climits>
#include <cstdio>
#include <cstring>
#include <fstream>
#include <string>
#include <system_error>
#include <thread>

#include <linux/futex.h>
#include <sched.h>
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

int processors_of_quota(const char *cpu_max) {
    long long quota = 0, period = 0;
    if (sscanf(cpu_max, "%lld %lld", &quota, &period) != 2 || quota <= 0 || period <= 0) return 0;
    return (int)std::min<long long>((quota + period - 1) / period, 1 << 20);
}

static std::string first_line(const std::string &file) {
    std::ifstream in(file);
    std::string line;
    std::getline(in, line);
    return line;
}

int available_processors() {
    int count = std::max(1, (int)std::thread::hardware_concurrency());
    cpu_set_t bound;
    if (sched_getaffinity(0, sizeof(bound), &bound) == 0) count = std::min(count, std::max(1, CPU_COUNT(&bound)));
    auto limit = [&](const std::string &cpu_max) {
        const int most = processors_of_quota(cpu_max.c_str());
        if (most > 0) count = std::min(count, most);
    };
    std::ifstream groups("/proc/self/cgroup");
    for (std::string line; std::getline(groups, line);) {
        const size_t first = line.find(':'), second = line.find(':', first + 1);
        if (second == std::string::npos) continue;
        const std::string controllers = line.substr(first + 1, second - first - 1);
        std::string path = line.substr(second + 1);
        const bool unified = controllers.empty();
        if (!unified && ("," + controllers + ",").find(",cpu,") == std::string::npos) continue;
        for (;;) {   // a limit anywhere above counts
            if (path == "/") path.clear();
            if (unified) {
                limit(first_line("/sys/fs/cgroup" + path + "/cpu.max"));
            } else {
                const std::string at = "/sys/fs/cgroup/cpu" + path;
                limit(first_line(at + "/cpu.cfs_quota_us") + " " + first_line(at + "/cpu.cfs_period_us"));
            }
            if (path.empty()) break;
            path.erase(path.rfind('/') == std::string::npos ? 0 : path.rfind('/'));
        }
    }
    return count;
}

void HostCopier::set_threads(int count) { limit_.store(count <= 0 ? std::min(kMost, std::max(1, available_processors() * 3 / 4)) : std::min(count, kMost)); }

int HostCopier::threads() {
    if (limit_.load() == 0) set_threads(0);
    return limit_.load();
}

void HostCopier::start() {
    try {
        for (; started_ < threads(); started_++) std::thread([this, i = started_]() { worker(i); }).detach();
    } catch (const std::system_error &) {   // no more threads to be had: the ones there are do
        limit_.store(started_);
    }
}

void HostCopier::worker(int index) {
    using clock = std::chrono::steady_clock;
    const bool near = index <= kNear;
    std::atomic<unsigned> &calls = near ? near_calls_ : far_calls_;
    std::atomic<int> &asleep = near ? near_asleep_ : far_asleep_;
    unsigned seen = 0;
    for (;;) {
        const unsigned call = calls.load();
        unsigned now = generation_.load();
        if (now == seen && near && index < limit_.load()) {
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
        if (index >= limit_.load()) continue;
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
    if (started_ < limit_.load() || limit_.load() == 0) start();
    near_calls_.fetch_add(1);
    if (near_asleep_.load() > 0) futex_wake(near_calls_);
}

void HostCopier::parallel(int pieces, bool large, const std::function<void(int)> &body, const std::function<void()> *idle) {
    if (pieces <= 1) {
        if (pieces == 1) body(0);
        if (idle != nullptr) (*idle)();
        return;
    }
    if (started_ < limit_.load() || limit_.load() == 0) start();
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
