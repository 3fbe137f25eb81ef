"""Host threads of the library (csrc/fs_threads.h) where the system refuses some or
all of them: every share is run, once, and the process goes on.  A small program
includes the header and takes pthread_create's place."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "finetoolsflexstructures.jl_amd", "csrc")

PROGRAM = r"""
#include "fs_threads.h"
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>
#include <atomic>
#include <cstdio>
#include <functional>
#include <stdexcept>
static std::atomic<int> left{0}, refused{0};
extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *x) noexcept {
    if (left-- <= 0) { ++refused; return EAGAIN; }
    static auto real = (int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *))dlsym(RTLD_NEXT, "pthread_create");
    return real(t, a, f, x);
}
int main() {
    for (int allowed : {0, 1, 3, 1000}) {
        for (int64_t n : {0, 1, 7, 100, 4096, 100000}) {
            left = allowed;
            std::vector<std::atomic<int>> hits(n);
            fs::parallel_chunks(n, [&](int64_t a, int64_t b) { for (int64_t i = a; i < b; ++i) ++hits[i]; }, 10);
            for (auto &h : hits) if (h != 1) return 1;
            left = allowed;
            std::atomic<int64_t> sum{0};
            fs::run_shares(n % 50, [&](int64_t t) { sum += t + 1; });
            if (sum != (n % 50) * (n % 50 + 1) / 2) return 2;
        }
        left = allowed;  // recursive halving, as the planners cut
        std::vector<std::atomic<int>> hits(5000);
        std::function<void(int64_t, int64_t)> halve = [&](int64_t b, int64_t n) {
            if (n <= 3) { for (int64_t i = b; i < b + n; ++i) ++hits[i]; return; }
            fs::run_shares(2, [&](int64_t t) { t ? halve(b + n / 2, n - n / 2) : halve(b, n / 2); });
        };
        halve(0, 5000);
        for (auto &h : hits) if (h != 1) return 3;
        left = allowed;  // an exception of the caller's own share finds the threads joined
        std::atomic<int> done{0};
        try {
            fs::run_shares(4, [&](int64_t t) { if (t == 0) throw std::runtime_error("x"); ++done; });
            return 4;
        } catch (const std::runtime_error &) {
            if (done != 3) return 5;
        }
    }
    std::printf("refused %d\n", refused.load());
    return refused > 0 ? 0 : 6;
}
"""


@pytest.mark.parametrize("threads", ["1", "4"])
def test_refused_threads(tmp_path, threads):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-rdynamic", "-pthread", "-I", CSRC, "-o", str(exe), str(src), "-ldl"],
                   check=True)
    r = subprocess.run([str(exe)], env=dict(os.environ, OMP_NUM_THREADS=threads), stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout)
