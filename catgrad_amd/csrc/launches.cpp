// The thread that passes a backend's launches on (launches.hpp).
#include "launches.hpp"

#include <sched.h>
#include <unistd.h>

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
    pid_t process = 0;
};
Open &open_queues() {
    static Open *const o = new Open;
    return *o;
}
void end_of_process() {
    Open &o = open_queues();
    if (getpid() != o.process) return; // (a forked child has none of the threads)
    std::lock_guard<std::mutex> lk(o.mu);
    for (LaunchQueue *q : o.all) q->end();
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
    if (!o.process) { // (behind the runtime's first call: what that leaves for the end of the process comes after this)
        o.process = getpid();
        (void)atexit(end_of_process);
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
    if (thread_.joinable()) {
        {
            std::lock_guard<std::mutex> lk(mu_);
            stop_ = true;
        }
        cv_.notify_one();
        thread_.join();
    }
    if (stream_) (void)hipStreamDestroy(stream_);
    stream_ = nullptr;
}

void LaunchQueue::wake() {
    {
        std::lock_guard<std::mutex> lk(mu_);
        awake_.store(true);
    }
    if (thread_.joinable()) {
        cv_.notify_one();
        return;
    }
    // (here, where the thread takes over what the caller is bound to)
    if (usable_cores() >= 2) {
        try {
            thread_ = std::thread([this] { work(); });
            return;
        } catch (const std::system_error &) {
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

void LaunchQueue::work() {
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
            std::this_thread::yield();
            continue;
        }
        std::unique_lock<std::mutex> lk(mu_);
        awake_.store(false);
        if (head_.load() != n) { // handed over in the meantime
            awake_.store(true);
            spins = 0;
            continue;
        }
        cv_.wait(lk, [this] { return awake_.load() || stop_; });
        if (stop_) return;
        spins = 0;
    }
}

} // namespace cg
