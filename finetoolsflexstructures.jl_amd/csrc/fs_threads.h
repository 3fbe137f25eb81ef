// fs_threads.h -- host threads of the planners and copies.  They live within one
// call, and a call whose threads the system refuses (a limit on processes, no memory
// for a stack) does their work on the threads that it has.
#pragma once
#include <sched.h>

#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <system_error>
#include <thread>
#include <utility>
#include <vector>

namespace fs {

// Host threads for the parallel loops: the CPUs this process may run on,
// capped by OMP_NUM_THREADS when that is set.
inline int64_t host_threads() {
    static const int64_t nt = [] {
        int64_t n = std::max<int64_t>(1, std::thread::hardware_concurrency());
        cpu_set_t set;
        if (sched_getaffinity(0, sizeof set, &set) == 0) n = std::max(1, CPU_COUNT(&set));
        if (const char *e = std::getenv("OMP_NUM_THREADS")) {
            const long v = std::strtol(e, nullptr, 10);
            if (v > 0) n = std::min<int64_t>(n, v);
        }
        return n;
    }();
    return nt;
}

// Threads joined at the end of their scope, also when that is left by an exception.
class Threads {
  public:
    ~Threads() {
        for (std::thread &t : th_) t.join();
    }
    // fn on a thread of its own; false if the system gives none
    template <class F>
    bool start(F fn) {
        th_.emplace_back();
        try {
            th_.back() = std::thread(std::move(fn));
            return true;
        } catch (const std::system_error &) {
            th_.pop_back();
            return false;
        }
    }

  private:
    std::vector<std::thread> th_;
};

// fn(0) to fn(nt - 1), each on a thread of its own where one can be had.
template <class F>
void run_shares(int64_t nt, const F &fn) {
    Threads th;
    for (int64_t t = 1; t < nt; ++t)
        if (!th.start([&fn, t] { fn(t); })) fn(t);
    if (nt > 0) fn(0);
}

// Runs fn(begin, end) over [0, n) in up to host_threads() chunks of at
// least `grain` iterations; for host loops whose iterations write disjoint data.
template <class F>
void parallel_chunks(int64_t n, const F &fn, int64_t grain = 65536) {
    const int64_t nt = std::max<int64_t>(1, std::min<int64_t>(host_threads(), n / grain));
    run_shares(nt, [&](int64_t t) { fn(n * t / nt, n * (t + 1) / nt); });
}

}  // namespace fs
