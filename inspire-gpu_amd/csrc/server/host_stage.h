// A small crew that prepares a call's host data in order while the calling
// thread launches what is ready: items 0, 1, ... are taken in order by the
// caller and its helper threads, and the caller waits for a prefix of them.
// One crew per server, sized at its creation and joined at its end; a call
// holds the server's mutex, so one job runs at a time.
#pragma once
#include <atomic>
#include <condition_variable>
#include <functional>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

namespace inspire {

class HostStage {
public:
    explicit HostStage(size_t helpers, size_t max_items) : done_(new std::atomic<uint8_t>[max_items]) {
        threads_.reserve(helpers);
        try {
            for (size_t i = 0; i < helpers; i++) threads_.emplace_back([this] { help(); });
        } catch (...) {
            // no more threads to be had: a job goes with those there are, or
            // with its caller alone (leaving here would end the process,
            // whose threads nothing joins)
        }
    }
    ~HostStage() {
        {
            std::lock_guard<std::mutex> lk(m_);
            stop_ = true;
        }
        cv_.notify_all();
        for (auto& t : threads_) t.join();
    }
    HostStage(const HostStage&) = delete;

    // Start items [0, n); with `wake` the helpers take part.
    void begin(size_t n, std::function<void(size_t)> fn, bool wake) {
        for (size_t i = 0; i < n; i++) done_[i].store(0, std::memory_order_relaxed);
        {
            std::lock_guard<std::mutex> lk(m_);
            fn_ = std::move(fn);
            n_ = n;
            next_.store(0);
            failed_.store(false);
            open_ = wake && !threads_.empty();
            job_++;
        }
        if (open_) cv_.notify_all();
    }
    // Return once items [0, upto) are done or have failed, taking part. A
    // failure does not end the wait: what the caller has enqueued by then is
    // followed by the rest, and it learns of the failure from finish().
    void wait(size_t upto) {
        for (size_t i = 0; i < upto; i++)
            while (!done_[i].load(std::memory_order_acquire))
                if (!take()) std::this_thread::yield();
    }
    // Every item done and no helper inside the job any more; whether none of
    // them failed.
    bool finish() {
        wait(n_);
        std::unique_lock<std::mutex> lk(m_);
        open_ = false;
        idle_.wait(lk, [&] { return active_ == 0; });
        return !failed_.load();
    }

private:
    bool take() {
        const size_t i = next_.fetch_add(1);
        if (i >= n_) return false;
        try {
            fn_(i);
        } catch (...) {
            failed_.store(true);
        }
        done_[i].store(1, std::memory_order_release);
        return true;
    }
    void help() {
        std::unique_lock<std::mutex> lk(m_);
        uint64_t seen = 0;
        for (;;) {
            cv_.wait(lk, [&] { return stop_ || (open_ && job_ != seen); });
            if (stop_) return;
            seen = job_;
            active_++;
            lk.unlock();
            while (take()) {
            }
            lk.lock();
            if (--active_ == 0) idle_.notify_all();
        }
    }

    std::vector<std::thread> threads_;
    std::unique_ptr<std::atomic<uint8_t>[]> done_;
    std::mutex m_;
    std::condition_variable cv_, idle_;
    std::function<void(size_t)> fn_;
    size_t n_ = 0, active_ = 0;
    std::atomic<size_t> next_{0};
    std::atomic<bool> failed_{false};
    uint64_t job_ = 0;
    bool open_ = false, stop_ = false;
};

}  // namespace inspire
