// A few threads that share the pieces of a host copy.
//
// One thread copies at about 14 GB/s, a quarter of the host link's rate, so a
// frame in ordinary host memory spends most of its upload in the copy to the
// page-locked staging chunks.  The owner of a team opens a job of numbered
// pieces, releases pieces in order as their destination becomes free, works
// on pieces itself and closes the job; the helpers take pieces while a job is
// open and sleep otherwise, also within a job once no piece has been released
// for kIdle (a GPU busy with other work can hold a staging chunk for as long as
// that work takes).  A team without helpers is the plain copy.  One thread at a
// time may use a team.
#pragma once

#include <pthread.h>
#include <signal.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

namespace cjx {

class CopyTeam {
public:
    // At most `helpers` threads, fewer on machines with fewer processors or
    // when the system refuses one.
    explicit CopyTeam(unsigned int helpers) noexcept {
        const unsigned int cpus{std::thread::hardware_concurrency()};
        // The helpers inherit a mask that leaves the process's signals to its
        // own threads.
        sigset_t every, before;
        sigfillset(&every);
        const bool masked{pthread_sigmask(SIG_SETMASK, &every, &before) == 0};
        for (unsigned int i{0}; i < helpers && i + 1 < cpus; ++i) {
            try {
                threads_.emplace_back([this] { helper(); });
            } catch (...) {
                break;
            }
        }
        if (masked) {
            (void)pthread_sigmask(SIG_SETMASK, &before, nullptr);
        }
    }

    ~CopyTeam() {
        {
            const std::lock_guard<std::mutex> lock{mutex_};
            stop_ = true;
        }
        wake_.notify_all();
        for (std::thread& t : threads_) {
            t.join();
        }
    }

    CopyTeam(const CopyTeam&) = delete;
    CopyTeam& operator=(const CopyTeam&) = delete;

    // A job of pieces copy(0), copy(1), ...; `done` pieces are counted per
    // group of `group` pieces (at most kGroups groups).  The helpers are
    // woken if `shared`.
    static constexpr std::uint32_t kGroups = 1024;

    void open(std::uint32_t pieces, std::uint32_t group, std::function<void(std::uint32_t)> copy, bool shared) {
        {
            const std::lock_guard<std::mutex> lock{mutex_};
            copy_ = std::move(copy);
            pieces_ = pieces;
            group_ = group;
            next_.store(0);
            released_.store(0);
            for (std::uint32_t g{0}; g < (pieces + group - 1) / group; ++g) {
                done_[g].store(0);
            }
            open_ = true;
            ++job_;
        }
        if (shared && !threads_.empty()) {
            wake_.notify_all();
        }
    }

    // Pieces below `n` may be copied.
    void release(std::uint32_t n) {
        released_.store(n);
        wake_sleeping();
    }

    // Copies pieces until all of group g, which has been released, are done.
    void finish_group(std::uint32_t g) {
        const std::uint32_t first{g * group_};
        const std::uint32_t count{pieces_ - first < group_ ? pieces_ - first : group_};
        while (done_[g].load(std::memory_order_acquire) < count) {
            if (!take()) {
                __builtin_ia32_pause();
            }
        }
    }

    // Ends the job (pieces not taken yet are left out) once no helper is at
    // work on it.
    void close() {
        {
            const std::lock_guard<std::mutex> lock{mutex_};
            open_ = false;
        }
        next_.store(pieces_);
        wake_sleeping();
        while (busy_.load(std::memory_order_acquire) != 0) {
            __builtin_ia32_pause();
        }
    }

private:
    // How long a helper polls for the next piece of an open job: ten times what
    // a staging chunk of 512 KB takes to come free on an idle device (19 us), so
    // that only a held-up upload pays for a wake-up.
    static constexpr std::chrono::microseconds kIdle{200};

    // After a change to next_ or released_.  A helper counts itself into
    // sleeping_ before it looks at them for the last time, so one of the two
    // sees the other's write; the lock keeps the call out of the time between
    // that look and the wait.
    void wake_sleeping() {
        if (sleeping_.load() != 0) {
            { const std::lock_guard<std::mutex> lock{mutex_}; }
            wake_.notify_all();
        }
    }

    // One released piece, if any is left.
    bool take() {
        std::uint32_t i{next_.load()};
        do {
            if (i >= released_.load(std::memory_order_acquire) || i >= pieces_) {
                return false;
            }
        } while (!next_.compare_exchange_weak(i, i + 1));
        copy_(i);
        done_[i / group_].fetch_add(1, std::memory_order_release);
        return true;
    }

    void helper() {
        std::uint64_t seen{0};
        std::unique_lock<std::mutex> lock{mutex_};
        for (;;) {
            wake_.wait(lock, [&] { return stop_ || (open_ && job_ != seen); });
            if (stop_) {
                return;
            }
            seen = job_;
            busy_.fetch_add(1);
            lock.unlock();
            auto last{std::chrono::steady_clock::now()};  // this helper's last piece
            for (unsigned int polls{1}; next_.load() < pieces_; ++polls) {
                if (take()) {
                    last = std::chrono::steady_clock::now();
                    continue;
                }
                __builtin_ia32_pause();
                if (polls % 64 == 0 && std::chrono::steady_clock::now() - last >= kIdle) {
                    lock.lock();
                    sleeping_.fetch_add(1);
                    wake_.wait(lock, [&] {
                        const std::uint32_t i{next_.load()};
                        return i >= pieces_ || i < released_.load();
                    });
                    sleeping_.fetch_sub(1);
                    lock.unlock();
                    last = std::chrono::steady_clock::now();
                }
            }
            busy_.fetch_sub(1, std::memory_order_release);
            lock.lock();
        }
    }

    std::mutex mutex_;
    std::condition_variable wake_;
    bool stop_{false}, open_{false};
    std::uint64_t job_{0};
    std::function<void(std::uint32_t)> copy_;
    std::uint32_t pieces_{0}, group_{1};
    std::atomic<std::uint32_t> next_{0}, released_{0}, busy_{0}, sleeping_{0};
    std::atomic<std::uint32_t> done_[kGroups]{};
    std::vector<std::thread> threads_;  // last: started with every other member in place
};

}  // namespace cjx
