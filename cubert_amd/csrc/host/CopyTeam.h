#ifndef CUBERT_HOST_COPYTEAM_H
#define CUBERT_HOST_COPYTEAM_H

#include <sched.h>

#include <condition_variable>
#include <cstddef>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace cuBERT {

// Copies between host arrays by the caller's thread and a few helpers of its own.  One thread moves a large output out of
// page-locked memory at 28 to 30 GB/s, half of what the copy engine brings.  The helpers sleep between copies, end with the object, and are
// not needed: whoever is awake takes the next share, so a copy is whole also where no helper could be started.
class CopyTeam {
public:
    // (two of 0.5 MB each are no faster shared: the helpers have to wake up)
    static constexpr size_t kWorthSharing = 1 << 20;

    CopyTeam() = default;
    CopyTeam(const CopyTeam &) = delete;
    CopyTeam &operator=(const CopyTeam &) = delete;

    ~CopyTeam() {
        {
            std::lock_guard<std::mutex> lock(mutex);
            ending = true;
        }
        wake.notify_all();
        for (std::thread &t : helpers) t.join();
    }

    // to be called when large copies are coming, while there is something else to wait for
    void start() noexcept {
        if (started) return;
        started = true;
        try {
            const size_t most = processors();
            helpers.reserve(kHelpers);
            while (helpers.size() < kHelpers && helpers.size() + 1 < most) helpers.emplace_back([this] { help(); });
        } catch (...) {
            // (as many as could be had)
        }
    }

    // the same as memcpy
    void copy(void *dst, const void *src, size_t bytes) {
        if (bytes < kWorthSharing || helpers.empty()) {
            std::memcpy(dst, src, bytes);
            return;
        }
        std::unique_lock<std::mutex> lock(mutex);
        to = static_cast<unsigned char *>(dst), from = static_cast<const unsigned char *>(src), left = bytes;
        wake.notify_all();
        take_shares(lock);
        done.wait(lock, [this] { return under_way == 0; });
    }

private:
    static constexpr size_t kHelpers = 3, kShare = 256 << 10;

    // that this thread, and with it its helpers, may run on (a container's share of time is not known here: helpers that get none are
    // not waited for, except for a share that they have taken)
    static size_t processors() {
        cpu_set_t set;
        if (sched_getaffinity(0, sizeof(set), &set) == 0) return (size_t) CPU_COUNT(&set);
        return std::thread::hardware_concurrency();
    }

    // shares of the current copy until there are none left; the lock is held on entry and on return
    void take_shares(std::unique_lock<std::mutex> &lock) {
        while (left > 0) {
            const size_t bytes = left < kShare ? left : kShare;
            unsigned char *dst = to;
            const unsigned char *src = from;
            to += bytes, from += bytes, left -= bytes;
            ++under_way;
            lock.unlock();
            std::memcpy(dst, src, bytes);
            lock.lock();
            if (--under_way == 0 && left == 0) done.notify_all();
        }
    }

    void help() {
        std::unique_lock<std::mutex> lock(mutex);
        while (!ending) {
            take_shares(lock);
            wake.wait(lock, [this] { return ending || left > 0; });
        }
    }

    std::mutex mutex;
    std::condition_variable wake, done;
    unsigned char *to = nullptr;
    const unsigned char *from = nullptr;
    size_t left = 0;       // of the current copy, not yet taken by anybody
    size_t under_way = 0;  // shares taken and not yet copied
    bool ending = false, started = false;
    std::vector<std::thread> helpers;
};

}  // namespace cuBERT

#endif  // CUBERT_HOST_COPYTEAM_H
