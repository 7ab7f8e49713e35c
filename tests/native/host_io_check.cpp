// Host-side check of the copy team (no GPU), run by tests/test_host_io.py:
//   1. copies of any size and number arrive whole;
//   2. a process forked from one whose team has helpers copies and destroys the team: the helpers are
//      not its own, and it neither waits for them nor ends by them;
//   3. nor when it destroys the team without a copy;
//   4. the pool keeps at most kIdleIos of what contexts leave, gives all back with the last of them, and
//      needs no memory to do so;
//   5. pinned memory is taken once the calls without it have paid for it, and at once where it is there
//      or small.
#include <cstdio>
#include <cstdlib>
#include <sys/wait.h>

#include "../../lightmetrica_amd/csrc/host_io.hpp"

using namespace lmgpu;

static bool no_memory = false;
__attribute__((noinline)) void* operator new(size_t n) {
    void* p = no_memory ? nullptr : std::malloc(n);
    if (!p) throw std::bad_alloc();
    return p;
}
__attribute__((noinline)) void operator delete(void* p) noexcept { std::free(p); }
__attribute__((noinline)) void operator delete(void* p, size_t) noexcept { std::free(p); }

static bool pool_gives_back() {
    HostIoPool pool;
    HostIo* ios[kIdleIos + 3];
    HostIo* gone[kIdleIos + 1];
    bool ok = true;
    size_t freed = 0;
    for (HostIo*& io : ios) {
        pool.context();
        ok = ok && (io = pool.acquire()) != nullptr;
    }
    ios[0]->bytes = kIdlePinned + 1;
    no_memory = true;
    try {
        for (HostIo* io : ios) {
            const size_t n = pool.release(io, gone);
            for (size_t k = 0; k < n; k++) delete gone[k];
            freed += n;
            const bool last = io == ios[kIdleIos + 2];
            ok = ok && (last || n == (io == ios[0] || io == ios[kIdleIos + 1] ? 1u : 0u));
        }
    } catch (...) {
        ok = false;
    }
    no_memory = false;
    return ok && freed == kIdleIos + 3;
}

static bool copies(CopyTeam& team) {
    bool ok = true;
    for (size_t bytes : {size_t(1), size_t(1000), size_t(512) << 10, (size_t(512) << 10) + 1, (size_t(9) << 20) + 17}) {
        std::vector<char> a(bytes), b(bytes + 2, 7), c(bytes / 3 + 1), d(bytes / 3 + 1, 9);
        for (size_t i = 0; i < bytes; i++) a[i] = char(i * 31 + (i >> 9));
        for (size_t i = 0; i < c.size(); i++) c[i] = char(i * 13 + 5);
        const CopyJob jobs[2] = {{b.data() + 1, a.data(), bytes}, {d.data(), c.data(), c.size()}};
        team.run(jobs, 2);
        ok = ok && std::memcmp(a.data(), b.data() + 1, bytes) == 0 && b[0] == 7 && b[bytes + 1] == 7 && c == d;
    }
    return ok;
}

static bool pays_in_time() {
    const size_t mib = size_t(1) << 20;
    HostIo io;
    bool ok = io.pays(HostIo::kPinAtOnce, 0.0);
    // 8 MiB for calls that save 400 us each: 3120 us, the eighth call's.
    for (int k = 1; k <= 8; k++) ok = ok && io.pays(8 * mib, 400.0) == (k == 8);
    ok = ok && !io.pays(8 * mib, 400.0);  // not had, for want of memory: asked for again as seldom
    io.bytes = 8 * mib;
    ok = ok && io.pays(8 * mib, 0.0) && io.pays(3 * mib, 0.0);
    HostIo streams;  // with 7000 us to prepare besides, then without
    streams.bytes = 8 * mib;
    for (int k = 1; k <= 7; k++) ok = ok && streams.pays(8 * mib, 1000.0, 7000.0) == (k == 7);
    ok = ok && streams.pays(8 * mib, 1.0);
    HostIo large;  // a call that pays for it by itself
    return ok && large.pays(8 * mib, 4000.0);
}

// Runs `child` in a forked process of a few seconds at most; its exit status, or -1 if a signal ended it.
template <class F> static int forked(F&& child) {
    std::fflush(stdout);
    const pid_t pid = fork();
    if (pid == 0) {
        alarm(5);
        _exit(child());
    }
    int status = 0;
    waitpid(pid, &status, 0);
    return WIFEXITED(status) ? WEXITSTATUS(status) : -1;
}

int main() {
    int failures = 0;
    CopyTeam* team = new CopyTeam;
    for (int k = 0; k < 8; k++)
        if (!copies(*team)) failures++, std::printf("copies differ\n");
    if (forked([&] {
            const bool ok = copies(*team);
            delete team;
            return ok ? 0 : 2;
        }) != 0)
        failures++, std::printf("a forked process that copied did not end well\n");
    if (forked([&] {
            delete team;
            return 0;
        }) != 0)
        failures++, std::printf("a forked process that did not copy did not end well\n");
    if (!copies(*team)) failures++, std::printf("copies differ after the forks\n");
    delete team;
    if (!pool_gives_back()) failures++, std::printf("the pool keeps or loses something\n");
    if (!pays_in_time()) failures++, std::printf("pinned memory is taken too early or too late\n");
    std::printf(failures ? "host_io_check: FAILED\n" : "host_io_check: OK\n");
    return failures ? 1 : 0;
}
