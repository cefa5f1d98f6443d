"""The queue between a backend and its launching thread (launches.hpp) on stand-ins for the runtime's calls: what a launch is given, in which order
launches are passed on, and what becomes of one that fails.  No GPU: a "kernel" is a plain function that the stand-in calls."""
import os
import subprocess

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


def test_one_core(tmp_path):
    """A process that may use one core has every launch made by its caller."""
    passes(tmp_path, r"""
int main() {
    auto &q = *queue();
    for (int n = 0; n < 500; n++) launch(q, n);
    q.drain();
    bool ok = check(by_thread == 0, "no other thread");
    ok &= check(seen.size() == 500, "all launched");
    for (int n = 0; n < (int)seen.size(); n++) ok &= check(seen[n] == n, "in order");
    q.close();
    if (ok) printf("done\n");
    return !ok;
}
""", prefix=("taskset", "-c", str(min(os.sched_getaffinity(0)))))


@pytest.mark.skipif(len(os.sched_getaffinity(0)) < 2, reason="a process on one core has no other thread")
def test_threads_moved_to_one_core(tmp_path):
    """A wait lets the thread that it waits for have the core, in less than a scheduler's turn (0.6 ms of processor time a hand-over here)."""
    passes(tmp_path, r"""
#include <dirent.h>
#include <sched.h>
#include <time.h>
int main() {
    auto &q = *queue();
    for (int n = 0; n < 100; n++) launch(q, n);
    q.drain();
    if (by_thread == 0) return printf("done\n"), 0; // (its control group has less than two cores)
    cpu_set_t set, one;
    sched_getaffinity(0, sizeof set, &set);
    CPU_ZERO(&one);
    for (int c = 0; c < CPU_SETSIZE; c++)
        if (CPU_ISSET(c, &set)) {
            CPU_SET(c, &one);
            break;
        }
    DIR *d = opendir("/proc/self/task");
    while (dirent *e = readdir(d))
        if (int t = atoi(e->d_name)) sched_setaffinity(t, sizeof one, &one);
    closedir(d);
    timespec a, b;
    clock_gettime(CLOCK_PROCESS_CPUTIME_ID, &a);
    for (int i = 0; i < 200; i++) {
        launch(q, i);
        q.drain();
    }
    clock_gettime(CLOCK_PROCESS_CPUTIME_ID, &b);
    const double us = ((b.tv_sec - a.tv_sec) * 1e6 + (b.tv_nsec - a.tv_nsec) * 1e-3) / 200;
    printf("%.0f us of processor time a hand-over\n", us);
    const bool ok = check(us < 250, "the wait gives way");
    q.close();
    if (ok) printf("done\n");
    return !ok;
}
""")


@pytest.mark.parametrize("membership,files,most", [
    ("0::/\n", {"cpu.max": "max 100000"}, None),
    ("0::/\n", {"cpu.max": "150000 100000"}, 1.5),
    ("0::/a/b\n", {"a/cpu.max": "50000 100000", "a/b/cpu.max": "max 100000"}, 0.5),
    ("0::/not/here\n", {"cpu.max": "100000 100000"}, 1.0),
    ("5:memory:/a\n4:cpu,cpuacct:/a\n", {"cpu/a/cpu.cfs_quota_us": "25000", "cpu/a/cpu.cfs_period_us": "100000", "cpu/cpu.cfs_quota_us": "-1"}, 0.25),
    ("3:cpuset:/a\n", {"cpu/a/cpu.cfs_quota_us": "25000", "cpu/a/cpu.cfs_period_us": "100000"}, None),
    ("1:cpu:/\nnonsense\n0::x\n", {"cpu.max": "", "cpu/cpu.cfs_quota_us": "100000"}, None),
], ids=lambda v: str(v) if isinstance(v, (float, type(None))) else "")
def test_processor_time(tmp_path, membership, files, most):
    """The least that a control group of the process is given, up to its bound cores."""
    (tmp_path / "membership").write_text(membership)
    for name, text in files.items():
        (tmp_path / "mount" / name).parent.mkdir(parents=True, exist_ok=True)
        (tmp_path / "mount" / name).write_text(text + "\n")
    bound = len(os.sched_getaffinity(0))
    want = bound if most is None else min(most, bound)
    passes(tmp_path, r"""
int main() {
    const double got = cg::usable_cores("%s", "%s");
    if (check(got == %r, "cores")) printf("done\n");
    else printf("%%g\n", got);
    return 0;
}
""" % (tmp_path / "membership", tmp_path / "mount", float(want)))


@pytest.mark.parametrize("closed", [False, True])
def test_end_of_process(tmp_path, closed):
    """A process that ends with launches on their way has them made before the runtime goes, and none behind it."""
    passes(tmp_path, r"""
static void gone() {
    runtime_gone = 1;
    std::this_thread::sleep_for(std::chrono::milliseconds(20));
    if (seen.size() == 60) printf("done\n");
}
int main() {
    atexit(gone); // (the runtime's own, left there by its first call)
    auto &q = *queue(), &other = *queue();
    busy_us = 100;
    for (int n = 0; n < 60; n++) launch(q, n);
    if (%d) q.close();
    other.close();
    return 0;
}
""" % closed)


@pytest.mark.parametrize("asleep", [False, True])
@pytest.mark.parametrize("child", ["exit(7);", "q.drain(); launch(q, 1000); q.close(); delete &q; if (seen.empty() || seen.back() != 1000) _exit(8); exit(7);"],
                         ids=["ends", "closes"])
def test_forked_child(tmp_path, child, asleep):
    """A forked child has none of its parent's threads: it ends, or closes what it has inherited, without waiting for one; its launches are its own."""
    passes(tmp_path, r"""
#include <signal.h>
#include <sys/wait.h>
int main() {
    auto &q = *queue();
    busy_us = 1000;
    for (int n = 0; n < 60; n++) launch(q, n);
    if (%d) {
        q.drain();
        usleep(20000);
    }
    const pid_t child = fork();
    if (!child) {
        %s
    }
    int status = 0;
    pid_t ended = 0;
    for (int i = 0; i < 500 && !(ended = waitpid(child, &status, WNOHANG)); i++) usleep(10000);
    const bool ok = check(ended == child && WIFEXITED(status) && WEXITSTATUS(status) == 7, "the child's own end");
    if (!ok && !ended) kill(child, SIGKILL);
    for (int n = 60; n < 120; n++) launch(q, n);
    q.close();
    if (ok && check(seen.size() == 120, "the parent's launches")) printf("done\n");
    return !ok;
}
""" % (asleep, child))
