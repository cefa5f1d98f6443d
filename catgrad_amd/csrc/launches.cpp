// The thread that passes a backend's launches on (launches.hpp).
#include "launches.hpp"

#include <pthread.h>
#include <sched.h>

#include <algorithm>
#include <chrono>
#include <cstdlib>
#include <fstream>
#include <string>
#include <system_error>
#include <vector>

namespace cg {
namespace {

// The open queues of the process, for its end.  (Never destroyed: a thread may close one while the process ends.)
struct Open {
    std::mutex mu;
    std::vector<LaunchQueue *> all;
    bool watched = false;
};
Open &open_queues() {
    static Open *const o = new Open;
    return *o;
}
void end_of_process() {
    Open &o = open_queues();
    std::lock_guard<std::mutex> lk(o.mu);
    for (LaunchQueue *q : o.all) q->end();
}
void before_fork() { open_queues().mu.lock(); }
void behind_fork() { open_queues().mu.unlock(); }
void in_child() {
    for (LaunchQueue *q : open_queues().all) q->forked();
    behind_fork();
}

} // namespace

double usable_cores(const char *membership, const char *mount) {
    cpu_set_t set;
    double cores = sched_getaffinity(0, sizeof set, &set) == 0 ? std::max(CPU_COUNT(&set), 1) : 1e9; // (more cores than a set holds)
    std::ifstream groups(membership);
    for (std::string line; std::getline(groups, line);) { // "<hierarchy>:<controllers>:<path>"; the unified hierarchy names no controllers
        const size_t a = line.find(':'), b = a == std::string::npos ? a : line.find(':', a + 1);
        if (b == std::string::npos) continue;
        const std::string what = "," + line.substr(a + 1, b - a - 1) + ",", root = std::string(mount) + (what == ",," ? "" : "/cpu");
        if (what != ",," && what.find(",cpu,") == std::string::npos) continue;
        for (std::string path = line.substr(b + 1);;) { // (a group has no more than those around it; in a container the path may be another one's)
            const std::string at = root + (path == "/" ? "" : path);
            std::string quota;
            double given = 0, period = 0;
            if (what == ",,") std::ifstream(at + "/cpu.max") >> quota >> period; // "max <period>" or "<quota> <period>"
            else if (std::ifstream(at + "/cpu.cfs_quota_us") >> quota) std::ifstream(at + "/cpu.cfs_period_us") >> period;
            if ((given = atof(quota.c_str())) > 0 && period > 0) cores = std::min(cores, given / period); // (no limit: "max", -1)
            if (path.empty() || path == "/") break;
            const size_t cut = path.rfind('/');
            path.resize(cut == std::string::npos ? 0 : cut);
        }
    }
    return cores;
}

hipError_t LaunchQueue::open(int device) {
    device_ = device;
    if (const hipError_t e = hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking)) return e;
    const char *t = getenv("CG_LAUNCH_THREAD"); // CG_LAUNCH_THREAD=0: every launch is the caller's
    if (!(t && t[0] == '0')) slots_.reset(new (std::nothrow) Slot[kSlots]);
    Open &o = open_queues();
    std::lock_guard<std::mutex> lk(o.mu);
    if (!o.watched) { // (behind the runtime's first call: what that leaves for the end of the process comes after this)
        o.watched = true;
        (void)atexit(end_of_process);
        (void)pthread_atfork(before_fork, behind_fork, in_child);
    }
    o.all.push_back(this);
    return hipSuccess;
}

void LaunchQueue::close() {
    {
        Open &o = open_queues();
        std::lock_guard<std::mutex> lk(o.mu);
        o.all.erase(std::remove(o.all.begin(), o.all.end(), this), o.all.end());
    }
    drain();
    if (worker_) {
        {
            std::lock_guard<std::mutex> lk(worker_->mu);
            worker_->stop = true;
        }
        worker_->cv.notify_one();
        worker_->thread.join();
        worker_.reset();
    }
    if (stream_) (void)hipStreamDestroy(stream_);
    stream_ = nullptr;
}

void LaunchQueue::wake() {
    if (worker_) {
        {
            std::lock_guard<std::mutex> lk(worker_->mu);
            awake_.store(true);
        }
        worker_->cv.notify_one();
        return;
    }
    // (here, where the thread takes over what the caller is bound to)
    if (usable_cores() >= 2) {
        try {
            worker_.reset(new Worker);
            awake_.store(true);
            worker_->thread = std::thread([this, w = worker_.get()] { work(*w); });
            return;
        } catch (const std::system_error &) {
            worker_.reset();
        }
    }
    // no thread to be had, or no core for it: what was handed over is passed on here, and so is what follows
    while (done_.load() != head_.load()) {
        pass_on(slots_[done_.load() % kSlots]);
        done_.fetch_add(1);
    }
    awake_.store(false);
    slots_.reset();
}

void LaunchQueue::work(Worker &w) {
    constexpr auto kLinger = std::chrono::microseconds(300); // between a step's last launch and the next step's first
    (void)hipSetDevice(device_);
    uint64_t n = 0;
    auto idle = std::chrono::steady_clock::now();
    for (uint32_t spins = 1;; spins++) {
        if (head_.load(std::memory_order_acquire) != n) {
            pass_on(slots_[n % kSlots]);
            done_.store(++n, std::memory_order_release);
            spins = 0;
            continue;
        }
        __builtin_ia32_pause();
        if (spins == 1) idle = std::chrono::steady_clock::now();
        if (spins % 64) continue;
        if (std::chrono::steady_clock::now() - idle < kLinger) {
            if (spins % 512 == 0) std::this_thread::yield(); // (not between the launches of a step)
            continue;
        }
        std::unique_lock<std::mutex> lk(w.mu);
        awake_.store(false);
        if (head_.load() != n) { // handed over in the meantime
            awake_.store(true);
            spins = 0;
            continue;
        }
        w.cv.wait(lk, [&] { return awake_.load() || w.stop; });
        if (w.stop) return;
        spins = 0;
    }
}

} // namespace cg
