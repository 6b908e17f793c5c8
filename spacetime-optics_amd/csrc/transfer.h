/* transfer.h - large copies from the device to pageable host memory (host code).

   What bounds them: a frame's memory is the caller's, usually fresh pages (a new array), and the runtime
   copies through its own pinned buffers with one thread, so the copy runs at the rate at which one core
   faults pages in: 10 GB/s into fresh pages, 17 GB/s into warm ones, where the link carries 57 GB/s. Here
   the DMA fills pinned slots one after the other, and THREADS threads each move their share of every
   filled slot to the caller's pages while the next is on its way. Copies below MIN_BYTES, and into memory
   that is already pinned, go straight to the runtime; so do copies to the device, which it moves at 30
   GB/s (the same threads measured no faster).
   The threads are woken when the stream reaches the copy: whatever it has to do before, they sleep. They
   are awake when the first slot is filled, and from then on the slots fill at the link's rate and they wait by
   yielding. There are at most as many as
   the process has cores (affinity, and the control group's quota); with one or two the runtime's path is taken.
   One Transfer per device serves all of its contexts (16 MiB of pinned memory take milliseconds to get)
   and ends with the last of them; it runs one copy at a time, and a copy that finds it busy takes the
   runtime's path. Measured (MI355X, 16 host cores), runtime -> threads: 3 MiB into
   fresh pages 0.72 -> 0.35 ms, 16 MiB 1.57 -> 0.51, 64 MiB 6.26 -> 2.34; into warm pages 3 MiB 0.18 ->
   0.14, 64 MiB 3.8 -> 1.5. */
#pragma once
#include <hip/hip_runtime.h>
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstdio>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

class Transfer {
  public:
    static constexpr int THREADS = 8, SLOTS = 4;
    static constexpr size_t SLOT = size_t(4) << 20;
    static constexpr size_t MIN_BYTES = size_t(3) << 19;

    // the device's Transfer, made for its first context and gone with its last
    static std::shared_ptr<Transfer> of_device(int device) {
        static std::mutex mu;
        static std::map<int, std::weak_ptr<Transfer>> all;
        std::lock_guard<std::mutex> lock(mu);
        std::shared_ptr<Transfer> t = all[device].lock();
        if (!t) all[device] = t = std::make_shared<Transfer>();
        return t;
    }

    Transfer() = default;
    Transfer(const Transfer&) = delete;
    Transfer& operator=(const Transfer&) = delete;
    ~Transfer() {
        {
            std::lock_guard<std::mutex> lock(mu_);
            stop_ = true;
        }
        wake_.notify_all();
        for (std::thread& t : threads_) t.join();
        for (Slot& s : slots_) {   // no copy is in flight: each one has waited for its events
            if (s.filled) (void)hipEventDestroy(s.filled);
            if (s.mem) (void)hipHostFree(s.mem);
        }
        if (reached_) (void)hipEventDestroy(reached_);
    }

    // device -> host after the work on the stream, complete on return
    hipError_t to_host(void* dst, const void* src, size_t bytes, hipStream_t st) {
        std::unique_lock<std::mutex> turn(busy_, std::defer_lock);
        if (bytes < MIN_BYTES || is_pinned(dst) || !turn.try_lock() || !ready()) {
            const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st);
            return e != hipSuccess ? e : hipStreamSynchronize(st);
        }
        // four pieces of a copy that fits the slots, so that the last one's move is short
        const size_t piece = std::min(SLOT, ((bytes / SLOTS) | 0xffff) + 1);
        dst_ = (char*)dst;
        bytes_ = bytes;
        piece_ = piece;
        pieces_ = (bytes + piece - 1) / piece;
        for (Slot& s : slots_) s.moved.store(0, std::memory_order_relaxed);
        hipError_t err = hipSuccess;
        auto fill = [&](size_t i) {
            Slot& s = slots_[i % SLOTS];
            if (err == hipSuccess)
                err = hipMemcpyAsync(s.mem, (const char*)src + i * piece, length(i), hipMemcpyDeviceToHost, st);
            if (err == hipSuccess) err = hipEventRecord(s.filled, st);
        };
        err = hipEventRecord(reached_, st);
        for (size_t i = 0; i < std::min<size_t>(pieces_, SLOTS); ++i) fill(i);
        if (err == hipSuccess) err = hipEventSynchronize(reached_);
        if (err != hipSuccess) {   // the threads have not been woken
            (void)hipStreamSynchronize(st);
            return err;
        }
        filled_.store(0, std::memory_order_relaxed);
        {
            std::lock_guard<std::mutex> lock(mu_);
            left_ = count_ - 1;
            ++turn_;
        }
        wake_.notify_all();
        for (size_t i = 0; i < pieces_; ++i) {
            if (err == hipSuccess) err = hipEventSynchronize(slots_[i % SLOTS].filled);
            if (err != hipSuccess) failed_.store(true, std::memory_order_relaxed);   // then nothing more is moved
            filled_.store(i + 1, std::memory_order_release);
            move_share(0, i);
            if (i + SLOTS < pieces_) {   // the slot is free again when every thread has taken its share
                while (slots_[i % SLOTS].moved.load(std::memory_order_acquire) < count_) std::this_thread::yield();
                slots_[i % SLOTS].moved.store(0, std::memory_order_relaxed);
                fill(i + SLOTS);
            }
        }
        {
            std::unique_lock<std::mutex> lock(mu_);
            over_.wait(lock, [this] { return left_ == 0; });
        }
        failed_.store(false, std::memory_order_relaxed);
        if (err != hipSuccess) (void)hipStreamSynchronize(st);   // nothing is left in flight into the slots
        return err;
    }

  private:
    struct Slot {
        char* mem = nullptr;
        hipEvent_t filled = nullptr;
        std::atomic<int> moved{0};   // threads that have taken their share of the piece in it
    };

    static bool is_pinned(const void* p) {
        hipPointerAttribute_t a;
        if (hipPointerGetAttributes(&a, p) != hipSuccess) {
            (void)hipGetLastError();   // ordinary memory may be reported as an error
            return false;
        }
        return a.type != hipMemoryTypeUnregistered;
    }

    size_t length(size_t i) const { return std::min(piece_, bytes_ - i * piece_); }

    // thread t's share of piece i: whole pages of it
    void move_share(int t, size_t i) {
        Slot& s = slots_[i % SLOTS];
        const size_t n = length(i), share = ((n / (size_t)count_) | 0xfff) + 1;
        const size_t a = std::min(n, share * (size_t)t), b = std::min(n, a + share);
        if (a < b && !failed_.load(std::memory_order_relaxed)) std::memcpy(dst_ + i * piece_ + a, s.mem + a, b - a);
        s.moved.fetch_add(1, std::memory_order_release);
    }

    // cores this process may use: its affinity, and the quota of its control group where there is one
    static int cores() {
        cpu_set_t set;
        int n = sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : (int)std::thread::hardware_concurrency();
        if (std::FILE* f = std::fopen("/sys/fs/cgroup/cpu.max", "r")) {
            double quota, period;
            if (std::fscanf(f, "%lf %lf", &quota, &period) == 2 && period > 0.0)
                n = std::min(n, std::max(1, (int)(quota / period + 0.5)));
            std::fclose(f);
        }
        return n;
    }

    // slots and threads, made at the first large copy; false (and the plain path) if they cannot be had
    bool ready() {
        if (state_ != 0) return state_ > 0;
        state_ = -1;
        count_ = std::min(THREADS, cores());
        if (count_ <= 2) return false;
        if (hipEventCreateWithFlags(&reached_, hipEventDisableTiming) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        for (Slot& s : slots_)
            if (hipHostMalloc((void**)&s.mem, SLOT, hipHostMallocDefault) != hipSuccess ||
                hipEventCreateWithFlags(&s.filled, hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                return false;
            }
        try {
            for (int t = 1; t < count_; ++t) threads_.emplace_back([this, t] { loop(t); });
        } catch (...) {
            return false;   // the threads that did start wait for a copy that never comes, until the end
        }
        state_ = 1;
        return true;
    }

    // a worker makes no device calls: it moves its share of each piece once the piece is there
    void loop(int t) {
        unsigned long long seen = 0;
        for (;;) {
            {
                std::unique_lock<std::mutex> lock(mu_);
                wake_.wait(lock, [&] { return stop_ || turn_ != seen; });
                if (stop_) return;
                seen = turn_;
            }
            for (size_t i = 0; i < pieces_; ++i) {
                while (filled_.load(std::memory_order_acquire) <= i) std::this_thread::yield();
                move_share(t, i);
            }
            std::lock_guard<std::mutex> lock(mu_);
            if (--left_ == 0) over_.notify_one();
        }
    }

    std::mutex busy_;   // one copy at a time
    int count_ = 0;     // threads, the caller among them
    int state_ = 0;     // 0: not tried, 1: slots and threads are there, -1: the plain path
    hipEvent_t reached_ = nullptr;   // the stream's work before the copy
    Slot slots_[SLOTS];
    std::vector<std::thread> threads_;
    std::mutex mu_;
    std::condition_variable wake_, over_;
    unsigned long long turn_ = 0;
    int left_ = 0;
    bool stop_ = false;
    // the copy under way
    char* dst_ = nullptr;
    size_t bytes_ = 0, piece_ = 0, pieces_ = 0;
    std::atomic<size_t> filled_{0};
    std::atomic<bool> failed_{false};
};
