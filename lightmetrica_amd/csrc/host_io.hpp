// Host arrays of the caller: copies between them and the context's pinned memory.
#pragma once
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstring>
#include <mutex>
#include <thread>
#include <unistd.h>
#include <vector>

namespace lmgpu {

struct CopyJob {
    char* dst;
    const char* src;
    size_t bytes;
};

// Copies with up to kTeam host threads: one thread's memcpy is slower than the link, most of all
// into pages that the caller has not touched yet.  The helpers are started by copies of at least
// kShared bytes and stay until the team is destroyed; starting seven threads for each copy took
// 0.1 to 0.3 ms.  Called by one thread at a time.
class CopyTeam {
public:
    ~CopyTeam() {
        if (helpers_.empty()) return;
        if (getpid() != owner_) {  // a forked child has no such threads
            for (auto& t : helpers_) t.detach();
            return;
        }
        {
            std::lock_guard<std::mutex> lock(m_);
            quit_ = true;
        }
        wake_.notify_all();
        for (auto& t : helpers_) t.join();
    }

    void run(const CopyJob* jobs, int njobs) {
        size_t total = 0;
        for (int j = 0; j < njobs; j++) total += jobs[j].bytes;
        if (total < kShared || !start()) {
            for (int j = 0; j < njobs; j++) std::memcpy(jobs[j].dst, jobs[j].src, jobs[j].bytes);
            return;
        }
        {
            std::lock_guard<std::mutex> lock(m_);
            jobs_ = jobs;
            njobs_ = njobs;
            next_.store(0, std::memory_order_relaxed);
            open_ = true;
            call_++;
        }
        wake_.notify_all();
        work(jobs, njobs);
        std::unique_lock<std::mutex> lock(m_);
        open_ = false;  // a helper that wakes up later finds nothing to do
        idle_.wait(lock, [&] { return working_ == 0; });
    }

private:
    static constexpr unsigned kTeam = 8;
    static constexpr size_t kShared = size_t(512) << 10;  // below, waking the helpers costs more than it gives
    static constexpr size_t kPiece = size_t(256) << 10;

    // Two more helpers a copy until the team is whole: starting one takes some 20 us.
    bool start() {
        owner_ = getpid();
        const unsigned n = std::min(kTeam, std::max(1u, std::thread::hardware_concurrency())) - 1;
        try {
            for (unsigned t = 0; t < 2 && helpers_.size() < n; t++) helpers_.emplace_back([this] { helper(); });
        } catch (...) {
            // fewer helpers
        }
        return !helpers_.empty();
    }

    void work(const CopyJob* jobs, int njobs) {
        for (;;) {
            size_t p = next_.fetch_add(1, std::memory_order_relaxed);
            int j = 0;
            for (; j < njobs; j++) {
                const size_t pieces = (jobs[j].bytes + kPiece - 1) / kPiece;
                if (p < pieces) break;
                p -= pieces;
            }
            if (j == njobs) return;
            const size_t off = p * kPiece;
            std::memcpy(jobs[j].dst + off, jobs[j].src + off, std::min(kPiece, jobs[j].bytes - off));
        }
    }

    void helper() {
        unsigned long long seen = 0;
        std::unique_lock<std::mutex> lock(m_);
        for (;;) {
            wake_.wait(lock, [&] { return quit_ || call_ != seen; });
            if (quit_) return;
            seen = call_;
            if (!open_) continue;
            const CopyJob* jobs = jobs_;
            const int njobs = njobs_;
            working_++;
            lock.unlock();
            work(jobs, njobs);
            lock.lock();
            if (--working_ == 0) idle_.notify_one();
        }
    }

    std::vector<std::thread> helpers_;
    std::mutex m_;
    std::condition_variable wake_, idle_;
    const CopyJob* jobs_ = nullptr;
    int njobs_ = 0;
    std::atomic<size_t> next_{0};
    unsigned long long call_ = 0;
    unsigned working_ = 0;
    bool open_ = false, quit_ = false;
    pid_t owner_ = 0;
};

// What a context needs to move host arrays: pinned memory, its first kPinnedWords bytes for small
// results, and a team.  A destroyed context leaves it to the next one, since fresh pinned memory
// costs 0.4 ms a megabyte when the host first touches it: at most kIdleIos of them are kept, with
// up to kIdlePinned bytes each, and all are freed with the last context (host_io_release).
struct HostIo {
    void* pinned = nullptr;
    size_t bytes = 0;
    CopyTeam team;
};
constexpr size_t kPinnedWords = 256;
constexpr size_t kIdleIos = 4;
constexpr size_t kIdlePinned = size_t(64) << 20;
void host_io_context();  // a context is created
HostIo* host_io_acquire();  // nullptr if there is no memory for it
void host_io_release(HostIo* io);  // a context is destroyed; io may be nullptr

}  // namespace lmgpu
