// Copies shared out over threads (csrc/host_copier.h) whose pieces or whose work between the pieces fail.
#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <set>
#include <stdexcept>
#include <thread>
#include <vector>

#include "host_copier.h"

using ios::HostCopier;

static int failures = 0;
#define CHECK(condition)                                              \
    do {                                                              \
        if (!(condition)) {                                           \
            printf("line %d: %s\n", __LINE__, #condition);            \
            failures++;                                               \
        }                                                             \
    } while (0)

static void doze(int us) { std::this_thread::sleep_for(std::chrono::microseconds(us)); }

// the pool still shares out a copy in full
static void check_copies() {
    std::vector<char> from(3 << 20), to(3 << 20);
    for (size_t i = 0; i < from.size(); i++) from[i] = (char)(i * 2654435761u >> 13);
    HostCopier::get().copy(to.data(), from.data(), from.size());
    CHECK(memcmp(to.data(), from.data(), from.size()) == 0);
    std::atomic<int> done{0};
    std::vector<std::atomic<int>> times(97);
    for (auto &t : times) t.store(0);
    HostCopier::get().parallel(97, true, [&](int i) {
        times[i].fetch_add(1);
        done.fetch_add(1);
    });
    CHECK(done.load() == 97);
    for (auto &t : times) CHECK(t.load() == 1);
}

// who throws: 0 the calling thread between its pieces, 1 the calling thread in a piece, 2 a worker in a piece, 3 nobody
static void check_failure(int who, bool large) {
    const auto caller = std::this_thread::get_id();
    std::atomic<int> inside{0}, begun{0};
    bool threw = false;
    int looks = 0;
    const std::function<void()> idle = [&]() {
        looks++;
        if (who == 0 && looks == 2) throw std::runtime_error("between the pieces");
    };
    try {
        HostCopier::get().parallel(64, large, [&](int) {
            inside.fetch_add(1);
            begun.fetch_add(1);
            const bool mine = std::this_thread::get_id() == caller;
            doze(mine ? 300 : 900);
            const bool fail = (who == 1 && mine) || (who == 2 && !mine);
            inside.fetch_sub(1);
            if (fail) throw std::runtime_error("in a piece");
        }, &idle);
    } catch (const std::runtime_error &e) {
        threw = true;
    }
    CHECK(inside.load() == 0);
    CHECK(threw == (who != 3) || (who == 2 && HostCopier::get().threads() < 2));
    CHECK(threw ? begun.load() < 64 : begun.load() == 64);
    const int then = begun.load();
    doze(2000);
    CHECK(begun.load() == then);   // nobody begins a piece behind the caller's back
}

// the pool with another number of threads
static void check_threads(int count) {
    HostCopier::get().set_threads(count);
    std::mutex mutex;
    std::set<std::thread::id> seen;
    for (int round = 0; round < 5; round++) {
        if (round) doze(1000);   // the workers are asleep, or awake
        HostCopier::get().parallel(40, true, [&](int) {
            doze(200);
            std::lock_guard<std::mutex> lock(mutex);
            seen.insert(std::this_thread::get_id());
        });
    }
    CHECK((int)seen.size() <= HostCopier::get().threads());
    CHECK(count == 0 || (int)seen.size() <= count);
    CHECK(count != 1 || seen.size() == 1);
    check_copies();
}

int main() {
    CHECK(ios::processors_of_quota("max 100000") == 0);
    CHECK(ios::processors_of_quota("400000 100000") == 4);
    CHECK(ios::processors_of_quota("50000 100000") == 1);
    CHECK(ios::processors_of_quota("150000 100000") == 2);
    CHECK(ios::processors_of_quota("-1 100000") == 0);
    CHECK(ios::processors_of_quota("") == 0);
    CHECK(ios::available_processors() >= 1 && ios::available_processors() <= (int)std::thread::hardware_concurrency());
    check_copies();
    CHECK(HostCopier::get().threads() <= std::max(1, ios::available_processors() * 3 / 4));
    for (int count : {1, 3, 2, 0, 1, 7, 0}) check_threads(count);
    for (int round = 0; round < 12; round++)
        for (int who = 0; who < 4; who++) {
            check_failure(who, round % 2 == 0);
            if (who % 2) check_copies();
        }
    for (int i = 0; i < 300; i++) {   // one failure after the other
        try {
            HostCopier::get().parallel(16, true, [&](int piece) {
                if (piece == i % 16) throw std::runtime_error("in a piece");
            });
            CHECK(false);
        } catch (const std::runtime_error &) {
        }
    }
    check_copies();
    printf(failures ? "FAILED\n" : "OK\n");
    return failures ? 1 : 0;
}
