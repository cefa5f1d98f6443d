// A backend's stream, and the kernels that are launched on it.
//
// The runtime takes about 3 us of host time for a launch, a backend's own calls around it 5 us: of a decode step of 150 launches of a
// small model 1.25 ms, where its kernels take 0.8.  So a backend that launches many kernels between two waits of the host hands
// them to a thread of its own, which does nothing but pass them on, in order, while the calling thread goes on (SmolLM2-135M shape
// 1.25 -> 0.97 ms a step, Qwen3-0.6B shape 1.66 -> 1.42).  The thread sleeps while there is nothing to pass on, and a few launches do not wake
// it: waking takes longer than they do.  Two threads that wait for each other need two cores: a process that may use less launches
// everything itself, and whoever waits longer than a launch takes lets others have its core (SmolLM2-135M shape, 512 tokens and 16 steps on one
// core: 24.7 ms, 392 with the thread and waits that keep the core; on two or more 18.7 to 20.4).
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstdlib>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <tuple>
#include <type_traits>
#include <utility>

namespace cg {

// A turn of waiting for another thread; 512 of them take 20 us.
inline void wait_turn(uint32_t &turns) {
    if (++turns % 512) __builtin_ia32_pause();
    else std::this_thread::yield();
}
// Cores that the calling thread and what it starts may use: what it is bound to, and the processor time that its control groups are given
// (`membership` names them, `mount` is where they lie).
double usable_cores(const char *membership = "/proc/self/cgroup", const char *mount = "/sys/fs/cgroup");

class LaunchQueue {
  public:
    LaunchQueue() = default;
    LaunchQueue(const LaunchQueue &) = delete;
    LaunchQueue &operator=(const LaunchQueue &) = delete;
    hipError_t open(int device);
    void close(); // everything handed over is on the stream; the thread ends, the stream goes
    // The process ends with this queue open: what was handed over is on the stream, and from now on every launch is its caller's (the
    // runtime goes next, and the thread must not be in it by then).
    void end() {
        ended_.store(true);
        drain();
    }
    // In a forked child, which has none of its parent's threads: what was handed over is the parent's, and every launch its caller's.
    void forked() {
        ended_.store(true);
        awake_.store(false);
        done_.store(head_.load());
        (void)worker_.release(); // (never destroyed here: its thread waits in it, in the parent)
    }

    // The stream, for anything but launch_kernel: what has been handed over is on it by then.
    operator hipStream_t() {
        drain();
        return stream_;
    }
    void drain() {
        for (uint32_t turns = 0; done_.load(std::memory_order_acquire) != head_.load(std::memory_order_relaxed);) wait_turn(turns);
    }
    // The host has waited for the device: the launches up to the next time are counted anew.
    void waited() { direct_ = 0; }
    // What the first launch that was handed over and failed since the last call has come to, and its kernel (hipSuccess: none).  Known when
    // what was launched behind it is known to have run.
    hipError_t error(const void **kernel) {
        const hipError_t e = failed_.load(std::memory_order_acquire);
        if (e == hipSuccess) return e;
        *kernel = failed_kernel_;
        failed_.store(hipSuccess, std::memory_order_release);
        return e;
    }

    // One caller at a time (the backend's lock); the arguments are copied.
    template <class... P, class... A> void launch(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, A &&...a) {
        typedef Job<P...> J;
        static_assert(std::is_trivially_destructible<J>::value && alignof(J) <= 16, "kernel arguments are plain values");
        if constexpr (sizeof(J) <= sizeof(Slot::job)) {
            if (hands_over()) {
                const uint64_t n = head_.load(std::memory_order_relaxed);
                for (uint32_t turns = 0; n - done_.load(std::memory_order_acquire) >= kSlots;) wait_turn(turns);
                Slot &s = slots_[n % kSlots];
                new (s.job) J{kernel, grid, block, lds, std::tuple<std::decay_t<P>...>(std::forward<A>(a)...)};
                s.run = &J::run;
                s.kernel = reinterpret_cast<const void *>(kernel);
                head_.store(n + 1);          // (either this thread sees the other one asleep, or that one the launch)
                if (!awake_.load()) wake();
                return;
            }
        }
        drain();
        J j{kernel, grid, block, lds, std::tuple<std::decay_t<P>...>(std::forward<A>(a)...)};
        (void)J::run(&j, stream_); // (an error is the caller's hipGetLastError)
    }

  private:
    static constexpr uint64_t kSlots = 64;
    // launches that the host makes itself before it wakes the thread: fewer than a forward pass of one layer has
    static constexpr int kDirect = 12;
    struct Slot {
        hipError_t (*run)(void *job, hipStream_t);
        const void *kernel;
        alignas(16) unsigned char job[4096 + 128]; // (the arguments of a kernel are at most 4096 bytes)
    };
    template <class... P> struct Job {
        void (*kernel)(P...);
        dim3 grid, block;
        size_t lds;
        std::tuple<std::decay_t<P>...> args;
        static hipError_t run(void *p, hipStream_t stream) {
            Job &j = *static_cast<Job *>(p);
            return std::apply(
                [&](auto &...a) {
                    void *at[sizeof...(P) + 1] = {&a...};
                    return hipLaunchKernel(reinterpret_cast<const void *>(j.kernel), j.grid, j.block, at, j.lds, stream);
                },
                j.args);
        }
    };
    bool hands_over() {
        if (!slots_ || ended_.load(std::memory_order_acquire)) return false;
        if (awake_.load(std::memory_order_acquire)) return true;
        return ++direct_ > kDirect;
    }
    void wake();
    struct Worker;
    void work(Worker &w);
    void pass_on(Slot &s) {
        const hipError_t e = s.run(s.job, stream_);
        if (e == hipSuccess || failed_.load(std::memory_order_acquire) != hipSuccess) return; // (the first one is kept)
        failed_kernel_ = s.kernel;
        failed_.store(e, std::memory_order_release);
    }

    int device_ = 0;
    hipStream_t stream_ = nullptr;
    int direct_ = 0;                 // launches since the host last waited that it made itself
    std::unique_ptr<Slot[]> slots_;  // null: every launch is the caller's
    alignas(64) std::atomic<uint64_t> head_{0}; // launches handed over
    alignas(64) std::atomic<uint64_t> done_{0}; // launches passed on
    std::atomic<bool> awake_{false}, ended_{false};
    std::atomic<hipError_t> failed_{hipSuccess};
    const void *failed_kernel_ = nullptr; // (written in front of failed_)
    struct Worker {
        bool stop = false;           // (under mu)
        std::mutex mu;
        std::condition_variable cv;
        std::thread thread;
    };
    std::unique_ptr<Worker> worker_; // from the first launch that is handed over on
};

template <class... P, class... A> inline void launch_kernel(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, LaunchQueue &on, A &&...a) {
    on.launch(kernel, grid, block, lds, std::forward<A>(a)...);
}

} // namespace cg
