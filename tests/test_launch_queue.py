"""The queue between a backend and its launching thread (launches.hpp) on stand-ins for the runtime's calls: what a launch is given, in which order
launches are passed on, and what becomes of one that fails.  No GPU: a "kernel" is a plain function that the stand-in calls."""
import subprocess
import os

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "catgrad_amd", "csrc")

HARNESS = r"""
#include "launches.hpp"
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <sys/syscall.h>
#include <unistd.h>
#include <vector>

struct Args { int n; void *const *args; };
static std::vector<int> seen;
static std::atomic<int> busy_us{0}, by_thread{0}, runtime_gone{0};
static const int own = (int)syscall(SYS_gettid);
extern "C" {
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = (hipStream_t)1, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t) {
    if (runtime_gone) {
        printf("launched behind the runtime's end\n");
        fflush(stdout);
        _exit(3);
    }
    if ((int)syscall(SYS_gettid) != own) by_thread++;
    const auto t0 = std::chrono::steady_clock::now();
    while (std::chrono::steady_clock::now() - t0 < std::chrono::microseconds(busy_us.load()));
    const int n = *static_cast<int *>(args[0]);
    if (n < 0) return (hipError_t)-n;
    ((void (*)(int))f)(n);
    return hipSuccess;
}
}
static void put(int n) { seen.push_back(n); }
static void other(int) {}
static cg::LaunchQueue *queue() {
    auto *q = new cg::LaunchQueue;
    if (q->open(0)) _exit(2);
    return q;
}
static void launch(cg::LaunchQueue &q, int n, void (*k)(int) = put) { cg::launch_kernel(k, dim3(1), dim3(1), 0, q, n); }
static bool check(bool ok, const char *what) {
    if (!ok) printf("wrong: %s\n", what);
    return ok;
}
"""


def build(tmp_path, program):
    (tmp_path / "harness.cpp").write_text(HARNESS + program)
    exe = str(tmp_path / "harness")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I", CSRC, "-I", "/opt/rocm/include", "-o", exe,
                           str(tmp_path / "harness.cpp"), os.path.join(CSRC, "launches.cpp")])
    return exe


def passes(tmp_path, program, env=None, prefix=()):
    r = subprocess.run([*prefix, build(tmp_path, program)], env=dict(os.environ, **(env or {})), capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.endswith("done\n"), r.stdout + r.stderr


@pytest.mark.parametrize("thread", ["1", "0"])
def test_order_and_errors(tmp_path, thread):
    """The first of several errors is kept with its kernel, reported once, and what is launched behind it is passed on all the same."""
    passes(tmp_path, r"""
int main() {
    auto &q = *queue();
    bool ok = true;
    for (int n = 0; n < 500; n++) launch(q, n);
    q.drain();
    ok &= check(seen.size() == 500, "all launched");
    for (int n = 0; n < (int)seen.size(); n++) ok &= check(seen[n] == n, "in order");
    const void *k = nullptr;
    ok &= check(q.error(&k) == hipSuccess && !k, "no error");
    if (by_thread > 0) { // (what the caller launches itself is the caller's to check)
        launch(q, -700, other);
        launch(q, -9);
        launch(q, 500);
        q.drain();
        ok &= check(q.error(&k) == 700 && k == (const void *)other, "the first error and its kernel");
        ok &= check(q.error(&k) == hipSuccess, "once");
        ok &= check(seen.size() == 501, "what follows is launched");
        launch(q, -9);
        q.drain();
        ok &= check(q.error(&k) == 9 && k == (const void *)put, "a later error");
    }
    q.close();
    if (ok) printf("done\n");
    return !ok;
}
""", {"CG_LAUNCH_THREAD": thread})
