// Device memory kept between the calls of consecutive bars (host code; the allocator
// behind it is passed in, so that the host self-test runs it on the CPU).
//
// A bar makes an operator and frees it: 14 GB in 120 ms at 43,248 tets, FP64, nmax 5.
// The driver wipes freed device memory at about 36 GB/s here; bars that follow one
// another faster build up a backlog, for which an allocation then waits up to
// seconds.  Bars of one mesh in a row, FP64, ms, mean (longest): 43,248 tets, nmax 5
// 384 (4,187) with every block freed, 119 (128) with the large ones kept; 103 k, nmax 6
// 1,176 (5,387) and 306 (307); 201 k, nmax 6 2,219 (6,391) and 601 (1,189), though its
// blocks exceed the limit.
//
//  * Bounded: at most `limit` bytes a device; the blocks kept longest go first.
//  * Given back: a thread frees what no call took for `idle` seconds; a failed
//    allocation and trim() free all of it at once.
//  * Safe across threads and streams: whoever keeps a block has waited for the device,
//    as a free does, so that its next owner may use it on any stream.
#pragma once

#include <algorithm>
#include <chrono>
#include <condition_variable>
#include <cstddef>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#include <unistd.h>

namespace scadyn {

class DevicePool {
public:
    typedef void (*Free)(int device, void *p);
    DevicePool(Free f, double idle_s) : free_(f), idle_(std::chrono::duration_cast<Clock::duration>(std::chrono::duration<double>(idle_s))) {}
    ~DevicePool() { stop(); }

    // Ends the thread; from then on blocks are freed at once.  What is still kept the
    // driver takes back at the process's end.  A forked child has no such thread:
    // nothing to wait for.
    void stop() {
        if (reaper_.joinable() && pid_ != getpid()) return;
        {
            std::lock_guard<std::mutex> lk(mu_);
            stop_ = true;
        }
        cv_.notify_all();
        if (reaper_.joinable()) reaper_.join();
    }

    // the smallest kept block of at least n and at most an eighth more bytes, or null
    void *take(int device, size_t n, size_t *size) {
        std::lock_guard<std::mutex> lk(mu_);
        auto best = blocks_.end();
        for (auto b = blocks_.begin(); b != blocks_.end(); ++b)
            if (b->device == device && b->size >= n && b->size - n <= n / 8 &&
                (best == blocks_.end() || b->size < best->size))
                best = b;
        if (best == blocks_.end()) return nullptr;
        void *p = best->p;
        *size = best->size;
        blocks_.erase(best);
        return p;
    }

    // keeps an idle block; what exceeds the limit is freed, all of it after stop() or
    // where the thread or the list's memory cannot be had (never throws: objects call it
    // as they end)
    void keep(int device, void *p, size_t size, size_t limit) noexcept {
        std::vector<Block> out;
        try {
            std::lock_guard<std::mutex> lk(mu_);
            if (!stop_ && !reaper_.joinable()) {
                pid_ = getpid();
                reaper_ = std::thread([this] { reap(); });
            }
            blocks_.reserve(blocks_.size() + 1);
            out.reserve(blocks_.size() + 1);
            if (stop_) limit = 0;
            blocks_.push_back({device, p, size, Clock::now() + idle_});
            size_t sum = 0;
            for (const Block &b : blocks_) sum += b.device == device ? b.size : 0;
            for (size_t i = 0; i < blocks_.size() && sum > limit;) {  // oldest first
                if (blocks_[i].device != device) {
                    ++i;
                    continue;
                }
                sum -= blocks_[i].size;
                out.push_back(blocks_[i]);
                blocks_.erase(blocks_.begin() + (long)i);
            }
        } catch (const std::exception &) {  // before the block was listed
            free_(device, p);
            return;
        }
        cv_.notify_all();
        for (const Block &b : out) free_(b.device, b.p);
    }

    size_t kept(int device) {
        std::lock_guard<std::mutex> lk(mu_);
        size_t sum = 0;
        for (const Block &b : blocks_) sum += b.device == device ? b.size : 0;
        return sum;
    }

    // frees all that is kept on a device; false when there was nothing
    bool trim(int device) {
        std::vector<Block> out;
        {
            std::lock_guard<std::mutex> lk(mu_);
            auto mine = std::stable_partition(blocks_.begin(), blocks_.end(), [&](const Block &b) { return b.device != device; });
            out.assign(mine, blocks_.end());
            blocks_.erase(mine, blocks_.end());
        }
        for (const Block &b : out) free_(b.device, b.p);
        return !out.empty();
    }

private:
    typedef std::chrono::steady_clock Clock;
    struct Block {
        int device;
        void *p;
        size_t size;
        Clock::time_point until;
    };

    void reap() {
        std::unique_lock<std::mutex> lk(mu_);
        while (!stop_) {
            if (blocks_.empty()) {
                cv_.wait(lk);
                continue;
            }
            // blocks are in the order of their times
            const Clock::time_point until = blocks_.front().until;  // the list may move meanwhile
            if (Clock::now() < until) {
                cv_.wait_until(lk, until);
                continue;
            }
            const Block b = blocks_.front();
            blocks_.erase(blocks_.begin());
            lk.unlock();
            free_(b.device, b.p);
            lk.lock();
        }
    }

    Free free_;
    Clock::duration idle_;
    std::mutex mu_;
    std::condition_variable cv_;
    std::vector<Block> blocks_;
    std::thread reaper_;
    pid_t pid_ = 0;  // the process that the thread runs in
    bool stop_ = false;
};

// The process's pool.  Its thread ends before the driver's own clean-up (statics made
// first go last); the object stays, since objects that end later may still free
// memory and since a forked child could not destroy what its parent's thread waits on.
inline DevicePool &process_pool(DevicePool::Free f, double idle_s) {
    static DevicePool *const pool = new DevicePool(f, idle_s);
    static struct End {
        ~End() { pool->stop(); }
    } end;
    return *pool;
}

}  // namespace scadyn
