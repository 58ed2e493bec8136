// The ring of pinned memory that large downloads go through, and the threads behind it (transfer.hip). Nothing here but the
// HIP calls of one copy at a time, declared by whoever includes it.
#pragma once
#include <string.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <mutex>
#include <thread>
#include <vector>

namespace vx {

struct Mover {
    static constexpr int SLOTS = 16, MAX_WORKERS = 6;
    static constexpr size_t SLOT = (size_t)1 << 20;
    struct Piece {
        char *dst;
        const char *src;
        size_t bytes;
    };
    struct Job {
        std::vector<Piece> pieces;
        std::vector<std::atomic<char>> copied;
        std::atomic<int> next{0}, arrived{0};
        std::atomic<bool> failed{false};
        explicit Job(std::vector<Piece> p) : pieces(std::move(p)), copied(pieces.size()) {
            for (auto &c : copied) c.store(0);
        }
    };
    char *ring = nullptr;
    hipEvent_t events[SLOTS] = {};
    std::vector<std::thread> workers;
    std::mutex call, mu;  // one transfer at a time; the fields below
    std::condition_variable wake, left;
    Job *job = nullptr;
    uint64_t turn = 0;
    int inside = 0;
    bool stop = false;

    ~Mover() {
        {
            std::lock_guard<std::mutex> g(mu);
            stop = true;
        }
        wake.notify_all();
        for (auto &t : workers) t.join();
        for (hipEvent_t e : events)
            if (e) (void)hipEventDestroy(e);
        if (ring) (void)hipHostFree(ring);
    }
    // helpers: threads beside the caller, who copies as well; fewer, or none, where the system gives no more
    bool start(int helpers) {
        if (hipHostMalloc((void **)&ring, SLOTS * SLOT, hipHostMallocDefault) != hipSuccess) {
            ring = nullptr;
            return false;
        }
        for (hipEvent_t &e : events)
            if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                e = nullptr;
                return false;
            }
        try {
            for (int i = 0; i < helpers; i++) workers.emplace_back([this] { work(); });
        } catch (...) {
        }
        return true;
    }
    void copy(Job &j, int i) {
        memcpy(j.pieces[i].dst, ring + (size_t)(i % SLOTS) * SLOT, j.pieces[i].bytes);
        j.copied[i].store(1, std::memory_order_release);
    }
    // Copies the next piece if it has arrived.
    bool take_arrived(Job &j) {
        int i = j.next.load();
        while (i < j.arrived.load(std::memory_order_acquire))
            if (j.next.compare_exchange_weak(i, i + 1)) {
                copy(j, i);
                return true;
            }
        return false;
    }
    // Takes pieces as they arrive until none is left.
    void run(Job &j) {
        const int n = (int)j.pieces.size();
        for (;;) {
            const int i = j.next.fetch_add(1);
            if (i >= n) return;
            while (j.arrived.load(std::memory_order_acquire) <= i) {
                if (j.failed.load()) return;
                std::this_thread::yield();
            }
            copy(j, i);
        }
    }
    void work() {
        uint64_t seen = 0;
        std::unique_lock<std::mutex> l(mu);
        for (;;) {
            wake.wait(l, [&] { return stop || (job && turn != seen); });
            if (stop) return;
            seen = turn;
            Job *j = job;
            inside++;
            l.unlock();
            run(*j);
            l.lock();
            if (--inside == 0) left.notify_all();
        }
    }
    // Everything before on the stream is done when this returns.
    hipError_t move(hipStream_t stream, Job &j) {
        const int n = (int)j.pieces.size();
        hipError_t err = hipSuccess;
        int sent = 0;
        for (int got = 0; got < n && err == hipSuccess; got++) {
            while (sent < n && err == hipSuccess) {
                if (sent >= SLOTS) {  // the slot's last piece has to be out of it; it has arrived, and may be nobody else's to copy
                    while (sent == got && !j.copied[sent - SLOTS].load(std::memory_order_acquire))
                        if (!take_arrived(j)) std::this_thread::yield();
                    if (!j.copied[sent - SLOTS].load(std::memory_order_acquire)) break;
                }
                const Piece &p = j.pieces[sent];
                err = hipMemcpyAsync(ring + (size_t)(sent % SLOTS) * SLOT, p.src, p.bytes, hipMemcpyDeviceToHost, stream);
                if (err == hipSuccess) err = hipEventRecord(events[sent % SLOTS], stream);
                sent++;
            }
            if (err == hipSuccess) err = hipEventSynchronize(events[got % SLOTS]);
            if (err != hipSuccess) break;
            j.arrived.store(got + 1, std::memory_order_release);
            if (got == 0) {  // (the threads sleep through the work that the first piece waits for)
                {
                    std::lock_guard<std::mutex> g(mu);
                    job = &j;
                    turn++;
                }
                wake.notify_all();
            }
        }
        if (err != hipSuccess) j.failed.store(true);
        else run(j);
        std::unique_lock<std::mutex> l(mu);
        job = nullptr;
        left.wait(l, [&] { return inside == 0; });
        return err;
    }
};

}  // namespace vx
