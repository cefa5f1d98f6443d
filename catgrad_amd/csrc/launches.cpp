// The thread that passes a backend's launches on (launches.hpp).
#include "launches.hpp"

#include <chrono>
#include <system_error>

namespace cg {

hipError_t LaunchQueue::open(int device) {
    device_ = device;
    if (const hipError_t e = hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking)) return e;
    const char *t = getenv("CG_LAUNCH_THREAD"); // CG_LAUNCH_THREAD=0: every launch is the caller's
    if (!(t && t[0] == '0')) slots_.reset(new (std::nothrow) Slot[kSlots]);
    return hipSuccess;
}

void LaunchQueue::close() {
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
    try {
        thread_ = std::thread([this] { work(); });
    } catch (const std::system_error &) { // no thread to be had: what was handed over is passed on here, and so is what follows
        while (done_.load() != head_.load()) {
            pass_on(slots_[done_.load() % kSlots]);
            done_.fetch_add(1);
        }
        awake_.store(false);
        slots_.reset();
    }
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
        if (spins % 64 || std::chrono::steady_clock::now() - idle < kLinger) continue;
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
