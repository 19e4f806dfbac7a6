// Host threads that share out a sequence of chunks, each as it becomes ready.
#pragma once

#include <condition_variable>
#include <cstdint>
#include <functional>
#include <mutex>
#include <thread>
#include <utility>
#include <vector>

namespace sev {

// part(chunk, t, nt) is thread t's share of a chunk among nt; it must not throw.
// As many threads as can be started, up to `want`; without any the shares run in
// publish(), on the calling thread.  (Thread: std::thread, or a stand-in whose
// constructor throws as std::thread's does.)
template <class Thread = std::thread>
class ChunkTeam {
   public:
    ChunkTeam(int want, int64_t chunks, std::function<void(int64_t, int, int)> part)
        : part_(std::move(part)), left_((size_t)chunks, 0) {
        th_.reserve((size_t)want);
        try {
            for (int t = 0; t < want; ++t) th_.emplace_back([this, t] { work(t); });
        } catch (...) {  // go on with those that run
        }
        // read by the threads only once a chunk is ready
        for (int &x : left_) x = (int)th_.size();
    }
    ChunkTeam(const ChunkTeam &) = delete;
    ChunkTeam &operator=(const ChunkTeam &) = delete;
    ~ChunkTeam() {
        {
            std::lock_guard<std::mutex> l(mu_);
            stop_ = true;
        }
        cv_.notify_all();
        for (auto &x : th_) x.join();
    }
    int size() const { return (int)th_.size(); }
    // chunk c is ready (in order)
    void publish(int64_t c) {
        if (th_.empty()) {
            part_(c, 0, 1);
            return;
        }
        {
            std::lock_guard<std::mutex> l(mu_);
            ready_ = c + 1;
        }
        cv_.notify_all();
    }
    // until every share of chunk c (published) has run
    void wait(int64_t c) {
        std::unique_lock<std::mutex> l(mu_);
        cv_.wait(l, [&] { return left_[(size_t)c] == 0; });
    }

   private:
    void work(int t) {
        for (int64_t c = 0; c < (int64_t)left_.size(); ++c) {
            {
                std::unique_lock<std::mutex> l(mu_);
                cv_.wait(l, [&] { return ready_ > c || stop_; });
                if (ready_ <= c) return;
            }
            part_(c, t, (int)th_.size());
            std::lock_guard<std::mutex> l(mu_);
            if (--left_[(size_t)c] == 0) cv_.notify_all();
        }
    }

    std::function<void(int64_t, int, int)> part_;
    std::mutex mu_;
    std::condition_variable cv_;
    int64_t ready_ = 0;      // chunks that are ready
    bool stop_ = false;      // no more will be
    std::vector<int> left_;  // shares of a chunk that have not run
    std::vector<Thread> th_;
};

}  // namespace sev
