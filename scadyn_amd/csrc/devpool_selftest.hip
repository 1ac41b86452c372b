// Host self-test of the device-memory pool (devpool.hpp) over a stand-in allocator:
// which block is taken, the limit, devices apart, memory given back after the idle
// time and on trim, threads that take and keep at once (no block ever has two
// owners, every block is freed once), a forked child that ends, objects freed
// after the pool's end, and a pool that cannot have its thread.
//
// Exit status 0 when all of it holds.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <random>
#include <set>

#include <csignal>
#include <pthread.h>
#include <sys/wait.h>
#include <unistd.h>

#include "devpool.hpp"

using namespace scadyn;

static int failures = 0, cases = 0;
static void expect(bool ok, const char *what) {
    ++cases;
    if (!ok) ++failures, std::printf("%s: FAIL\n", what);
}

static std::mutex g_mu;
static std::multiset<void *> g_freed;
static void fake_free(int, void *p) {
    std::lock_guard<std::mutex> lk(g_mu);
    g_freed.insert(p);
}
static size_t freed(void *p) {
    std::lock_guard<std::mutex> lk(g_mu);
    return g_freed.count(p);
}
static void *at(size_t i) { return (void *)(i * 64 + 64); }

// a user's static object that frees its memory after the pool's end: the child's exit
// status is 3 where that memory was freed
static struct Late {
    bool armed = false;
    ~Late() {
        if (!armed) return;
        process_pool(fake_free, 60.0).keep(0, at(21), 100, 1000);
        _exit(freed(at(21)) == 1 ? 3 : 4);
    }
} g_late;

// exit status of a child that runs f and ends as programs do; -1 where it hangs
template <class F>
static int child(F f) {
    std::fflush(stdout);
    const pid_t p = fork();
    if (p == 0) {
        f();
        std::exit(0);
    }
    for (int i = 0; i < 200; ++i) {
        int st = 0;
        if (waitpid(p, &st, WNOHANG) == p) return WIFEXITED(st) ? WEXITSTATUS(st) : -2;
        std::this_thread::sleep_for(std::chrono::milliseconds(50));
    }
    (void)kill(p, SIGKILL);
    (void)waitpid(p, nullptr, 0);
    return -1;
}

int main() {
    expect(child([] {
               process_pool(fake_free, 60.0).keep(0, at(20), 100, 1000);
               g_late.armed = true;
           }) == 3,
           "an object freed after the pool's end");
    {
        DevicePool pool(fake_free, 60.0);
        size_t size = 0;
        expect(!pool.take(0, 100, &size) && !pool.trim(0) && pool.kept(0) == 0, "empty pool");
        pool.keep(0, at(1), 1000, 10000);
        pool.keep(0, at(2), 1100, 10000);
        pool.keep(1, at(3), 1010, 10000);
        expect(pool.kept(0) == 2100 && pool.kept(1) == 1010, "kept bytes by device");
        expect(!pool.take(0, 1101, &size), "no block too small");
        expect(!pool.take(0, 880, &size), "no block more than an eighth too large");
        expect(pool.take(0, 1000, &size) == at(1) && size == 1000, "the smallest that fits");
        expect(pool.take(0, 1000, &size) == at(2) && size == 1100, "the next");
        expect(!pool.take(0, 1000, &size) && pool.kept(0) == 0, "another device's block stays");
        pool.keep(0, at(4), 4000, 9000);
        pool.keep(0, at(5), 4000, 9000);
        pool.keep(0, at(6), 4000, 9000);
        expect(freed(at(4)) == 1 && pool.kept(0) == 8000, "the oldest goes at the limit");
        pool.keep(0, at(7), 20000, 9000);
        expect(freed(at(5)) == 1 && freed(at(6)) == 1 && freed(at(7)) == 1 && pool.kept(0) == 0, "a block beyond the limit");
        expect(freed(at(3)) == 0 && pool.kept(1) == 1010, "the limit counts each device's own");
        expect(pool.trim(1) && freed(at(3)) == 1 && !pool.trim(1), "trim");
    }
    {
        DevicePool pool(fake_free, 0.05);
        pool.keep(0, at(10), 100, 1000);
        std::this_thread::sleep_for(std::chrono::milliseconds(30));
        pool.keep(0, at(11), 200, 1000);
        std::this_thread::sleep_for(std::chrono::milliseconds(400));
        expect(freed(at(10)) == 1 && freed(at(11)) == 1 && pool.kept(0) == 0, "given back after the idle time");
        pool.keep(0, at(12), 100, 1000);
        std::this_thread::sleep_for(std::chrono::milliseconds(400));
        expect(freed(at(12)) == 1, "and again");
    }
    {
        const int T = 6, N = 20000;
        DevicePool pool(fake_free, 0.002);
        std::atomic<size_t> next{1000};
        std::atomic<int> twice{0};
        std::mutex mu;
        std::set<void *> owned;  // blocks in some thread's hands
        std::vector<std::thread> th;
        for (int t = 0; t < T; ++t)
            th.emplace_back([&, t] {
                std::mt19937 rng(t);
                for (int i = 0; i < N; ++i) {
                    const size_t n = 100 + rng() % 50;
                    size_t size = n;
                    void *p = pool.take(t % 2, n, &size);
                    if (!p) p = at(next++);
                    {
                        std::lock_guard<std::mutex> lk(mu);
                        twice += !owned.insert(p).second;
                    }
                    if (freed(p)) ++twice;
                    {
                        std::lock_guard<std::mutex> lk(mu);
                        owned.erase(p);
                    }
                    pool.keep(t % 2, p, size, 800);
                    if (rng() % 500 == 0) pool.trim(t % 2);
                }
            });
        for (auto &x : th) x.join();
        pool.trim(0);
        pool.trim(1);
        std::this_thread::sleep_for(std::chrono::milliseconds(50));
        bool once = true;
        for (size_t i = 1000; i < next; ++i) once &= freed(at(i)) == 1;
        expect(twice == 0, "one owner at a time, none freed before");
        expect(once, "each block freed once");
    }
    {
        // threads' default stack larger than the address space: none can be made
        pthread_attr_t was, huge;
        (void)pthread_getattr_default_np(&was);
        pthread_attr_init(&huge);
        const bool set = pthread_attr_setstacksize(&huge, (size_t)1 << 50) == 0 && pthread_setattr_default_np(&huge) == 0;
        expect(set, "a stack size that no thread gets");
        DevicePool pool(fake_free, 60.0);
        if (set) pool.keep(0, at(23), 100, 1000);
        (void)pthread_setattr_default_np(&was);
        expect(freed(at(23)) == 1 && pool.kept(0) == 0, "freed at once without a thread");
        pool.keep(0, at(24), 100, 1000);
        expect(freed(at(24)) == 0 && pool.kept(0) == 100, "kept once there is one");
    }
    process_pool(fake_free, 60.0).keep(0, at(22), 100, 1000);
    std::this_thread::sleep_for(std::chrono::milliseconds(50));  // its thread waits
    expect(child([] {}) == 0, "a forked child ends");
    std::printf("%d cases, %d failures\n", cases, failures);
    return failures != 0;
}
