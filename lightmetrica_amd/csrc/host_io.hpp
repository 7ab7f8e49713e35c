// Host arrays of the caller: copies between them and the context's pinned memory.
#pragma once
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>
#include <type_traits>
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
// 0.1 to 0.3 ms.  Called by one thread at a time.  In a process forked from the one that started
// them there are no helpers: a team copies alone there and leaves what the helpers wait on as it is.
class CopyTeam {
public:
    ~CopyTeam() {
        if (!crew_ || getpid() != owner_) return;
        {
            std::lock_guard<std::mutex> lock(crew_->m);
            crew_->quit = true;
        }
        crew_->wake.notify_all();
        for (auto& t : crew_->helpers) t.join();
        delete crew_;
    }

    void run(const CopyJob* jobs, int njobs) {
        size_t total = 0;
        for (int j = 0; j < njobs; j++) total += jobs[j].bytes;
        if (total < kShared || !start()) {
            for (int j = 0; j < njobs; j++) std::memcpy(jobs[j].dst, jobs[j].src, jobs[j].bytes);
            return;
        }
        Crew& c = *crew_;
        {
            std::lock_guard<std::mutex> lock(c.m);
            c.jobs = jobs;
            c.njobs = njobs;
            c.next.store(0, std::memory_order_relaxed);
            c.open = true;
            c.call++;
        }
        c.wake.notify_all();
        c.work(jobs, njobs);
        std::unique_lock<std::mutex> lock(c.m);
        c.open = false;  // a helper that wakes up later finds nothing to do
        c.idle.wait(lock, [&] { return c.working == 0; });
    }

private:
    static constexpr unsigned kTeam = 8;
    static constexpr size_t kShared = size_t(512) << 10;  // below, waking the helpers costs more than it gives
    static constexpr size_t kPiece = size_t(256) << 10;

    // The helpers and what they share, on the heap: a forked process can destroy neither a thread that
    // it does not have nor a condition that such a thread waits on.
    struct Crew {
        std::vector<std::thread> helpers;
        std::mutex m;
        std::condition_variable wake, idle;
        const CopyJob* jobs = nullptr;
        int njobs = 0;
        std::atomic<size_t> next{0};
        unsigned long long call = 0;
        unsigned working = 0;
        bool open = false, quit = false;

        void work(const CopyJob* list, int n) {
            for (;;) {
                size_t p = next.fetch_add(1, std::memory_order_relaxed);
                int j = 0;
                for (; j < n; j++) {
                    const size_t pieces = (list[j].bytes + kPiece - 1) / kPiece;
                    if (p < pieces) break;
                    p -= pieces;
                }
                if (j == n) return;
                const size_t off = p * kPiece;
                std::memcpy(list[j].dst + off, list[j].src + off, std::min(kPiece, list[j].bytes - off));
            }
        }

        void help() {
            unsigned long long seen = 0;
            std::unique_lock<std::mutex> lock(m);
            for (;;) {
                wake.wait(lock, [&] { return quit || call != seen; });
                if (quit) return;
                seen = call;
                if (!open) continue;
                const CopyJob* list = jobs;
                const int n = njobs;
                working++;
                lock.unlock();
                work(list, n);
                lock.lock();
                if (--working == 0) idle.notify_one();
            }
        }
    };

    // Two more helpers a copy until the team is whole: starting one takes some 20 us.  False if there
    // is none.
    bool start() {
        if (!crew_) {
            crew_ = new (std::nothrow) Crew;
            owner_ = getpid();
        }
        if (!crew_ || getpid() != owner_) return false;
        Crew* const c = crew_;
        const unsigned n = std::min(kTeam, std::max(1u, std::thread::hardware_concurrency())) - 1;
        try {
            for (unsigned t = 0; t < 2 && c->helpers.size() < n; t++) c->helpers.emplace_back([c] { c->help(); });
        } catch (...) {
            // fewer helpers
        }
        return !c->helpers.empty();
    }

    Crew* crew_ = nullptr;
    pid_t owner_ = 0;
};

// What a context needs to move host arrays: pinned memory, its first kPinnedWords bytes for small
// results, and a team.  A destroyed context leaves it to the next one, since fresh pinned memory
// costs 0.39 ms a MiB when the host first touches it: at most kIdleIos of them are kept, with
// up to kIdlePinned bytes each, and all are freed with the last context (host_io_release).
struct HostIo {
    void* pinned = nullptr;
    size_t bytes = 0;
    CopyTeam team;

    // Whether a call that would save `saved_us` takes its way through `need` bytes of pinned memory,
    // which `more_us` of other preparation (0 once done) has to go before.  Fresh pinned pages cost the
    // host 0.39 ms a MiB (kTouchUs: 8 MiB 2.9 ms, 31 MiB 12.2), many times what one call saves, so calls
    // take the runtime's way until what they would have saved has paid for them: a program that renders
    // one image loses nothing, one that goes on never more than it spent.  First calls in a process
    // with all of it pinned at once, and before (us): a raycast of 1280 x 720 2600, 1040; 65000 rays
    // 1000, 510; 300,000 rays 13,000, 1380.  Up to kPinAtOnce the two are alike (10,000 rays 356, 358).
    bool pays(size_t need, double saved_us, double more_us = 0.0) {
        const bool fresh = need > bytes && need > kPinAtOnce;
        if (!fresh && more_us == 0.0) return true;
        saved_ += saved_us;
        if (saved_ < (fresh ? double(need) * (kTouchUs / (1 << 20)) : 0.0) + more_us) return false;
        saved_ = 0.0;
        return true;
    }

    static constexpr double kTouchUs = 390.0;  // a MiB
    static constexpr size_t kPinAtOnce = size_t(512) << 10;

private:
    double saved_ = 0.0;
};
constexpr size_t kPinnedWords = 256;
constexpr size_t kIdleIos = 4;
constexpr size_t kIdlePinned = size_t(64) << 20;
// The pool itself, which knows no HIP: release() hands back what is to be freed.  Nothing in it throws
// (a context is destroyed through a C entry), and it is trivially destroyed: contexts may be destroyed
// after static objects are.
class HostIoPool {
public:
    void context() {
        std::lock_guard<std::mutex> lock(m_);
        contexts_++;
    }
    HostIo* acquire() {  // nullptr if there is no memory for it
        std::lock_guard<std::mutex> lock(m_);
        return num_idle_ ? idle_[--num_idle_] : new (std::nothrow) HostIo;
    }
    // A context is destroyed; io may be nullptr.  Returns how many of `gone` are to be freed.
    size_t release(HostIo* io, HostIo* (&gone)[kIdleIos + 1]) {
        std::lock_guard<std::mutex> lock(m_);
        size_t n = 0;
        if (io && num_idle_ < kIdleIos && io->bytes <= kIdlePinned) idle_[num_idle_++] = io;
        else if (io) gone[n++] = io;
        if (--contexts_ == 0)
            while (num_idle_) gone[n++] = idle_[--num_idle_];
        return n;
    }

private:
    std::mutex m_;
    HostIo* idle_[kIdleIos] = {};
    size_t num_idle_ = 0, contexts_ = 0;
};
static_assert(std::is_trivially_destructible_v<HostIoPool>, "the pool outlives static objects");

void host_io_context();  // a context is created
HostIo* host_io_acquire();  // nullptr if there is no memory for it
void host_io_release(HostIo* io);  // a context is destroyed; io may be nullptr

}  // namespace lmgpu
