// Driver of csrc/host/CopyTeam.h for tests/test_copy_team.py: copies of many sizes and alignments by a team with as many helpers as the
// processor affinity (argv[1] processors; 0: as it is) and the thread library (argv[2] threads can be had; below 0: any number) allow.
#include <pthread.h>
#include <sched.h>

#include <cstdio>
#include <cstdlib>
#include <memory>
#include <vector>

#include "CopyTeam.h"

#ifdef COUNT_THREADS
#include <dlfcn.h>

#include <cerrno>
static int threads_left = -1, threads_started = 0;
extern "C" int pthread_create(pthread_t *thread, const pthread_attr_t *attr, void *(*run)(void *), void *arg) {
    if (threads_left == 0) return EAGAIN;
    if (threads_left > 0) --threads_left;
    ++threads_started;
    typedef int (*Create)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
    return reinterpret_cast<Create>(dlsym(RTLD_NEXT, "pthread_create"))(thread, attr, run, arg);
}
#endif

using cuBERT::CopyTeam;

static int failures = 0;
static void check(bool good, const char *what, size_t bytes) {
    if (good) return;
    ++failures;
    std::printf("FAILED %s, %zu bytes\n", what, bytes);
}

static void copies(CopyTeam &team, unsigned seed) {
    const size_t kMost = (5u << 20) + 4096, kGuard = 64;
    std::vector<unsigned char> from(kMost + kGuard), to(kMost + 2 * kGuard);
    for (size_t i = 0; i < from.size(); ++i) from[i] = (unsigned char) ((i * 2654435761u + seed) >> 13);
    const size_t share = 256 << 10, worth = CopyTeam::kWorthSharing;
    for (size_t bytes : {(size_t) 0, (size_t) 1, share, worth - 1, worth, worth + 1, 5 * share - 1, 5 * share + 3, (size_t) 4 << 20, kMost}) {
        const size_t at = seed % 3, off = seed % 5;
        std::fill(to.begin(), to.end(), (unsigned char) 0xa5);
        team.copy(to.data() + kGuard + off, from.data() + at, bytes);
        check(std::memcmp(to.data() + kGuard + off, from.data() + at, bytes) == 0, "contents", bytes);
        bool kept = true;
        for (size_t i = 0; i < kGuard + off; ++i) kept = kept && to[i] == 0xa5;
        for (size_t i = kGuard + off + bytes; i < to.size(); ++i) kept = kept && to[i] == 0xa5;
        check(kept, "bytes around", bytes);
    }
}

int main(int argc, char **argv) {
    const int processors = argc > 1 ? std::atoi(argv[1]) : 0, threads = argc > 2 ? std::atoi(argv[2]) : -1;
    if (processors > 0) {
        cpu_set_t allowed, some;
        sched_getaffinity(0, sizeof(allowed), &allowed);
        CPU_ZERO(&some);
        for (int cpu = 0, n = 0; cpu < CPU_SETSIZE && n < processors; ++cpu) {
            if (CPU_ISSET(cpu, &allowed)) CPU_SET(cpu, &some), ++n;
        }
        if (sched_setaffinity(0, sizeof(some), &some) != 0) return 2;
    }
#ifdef COUNT_THREADS
    threads_left = threads;
#endif
    {
        CopyTeam never_used, never_started;
        never_used.start();
        copies(never_started, 1);
    }
    for (unsigned seed = 0; seed < 4; ++seed) {  // ended with helpers asleep, and right behind a copy
        std::unique_ptr<CopyTeam> team(new CopyTeam);
        team->start();
        copies(*team, seed);
        team->start();
        copies(*team, seed + 7);
    }
    {  // a team per instance, from threads of their own
        std::vector<std::thread> callers;
        try {
            for (unsigned i = 0; i < 3; ++i) {
                callers.emplace_back([i] {
                    CopyTeam team;
                    team.start();
                    copies(team, 20 + i);
                });
            }
        } catch (...) {
        }
        for (std::thread &t : callers) t.join();
    }
#ifdef COUNT_THREADS
    std::printf("threads %d\n", threads_started);
#else
    (void) threads;
#endif
    if (failures == 0) std::printf("copy_team ok\n");
    return failures != 0;
}
