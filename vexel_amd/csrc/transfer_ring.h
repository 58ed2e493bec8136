// The ring of pinned memory that large downloads go through, and the threads behind it (transfer.hip). Nothing here but the
// HIP calls of one copy at a time, declared by whoever includes it; a kernel that sends many pieces at once comes from outside.
#pragma once
#include <string.h>
#include <sys/mman.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <mutex>
#include <thread>
#include <utility>
#include <vector>

namespace vx {

struct Mover {
    static constexpr int SLOTS = 16, MAX_WORKERS = 6;
    static constexpr size_t SLOT = (size_t)1 << 20;
    // With a sender the same ring has more and smaller slots, and a mark behind each that says which piece is in it.
    static constexpr int SENT_SLOTS = 256, SENT_MOST = 64, MARK_STEP = 8;  // (marks on cache lines of their own)
    static constexpr size_t SENT_SLOT = SLOTS * SLOT / SENT_SLOTS;
    struct Piece {
        char *dst;
        const char *src;
        size_t bytes;
    };
    struct Job {
        std::vector<Piece> pieces;
        std::vector<std::atomic<char>> copied;
        std::atomic<int> next{0}, arrived{0}, done{0};
        std::atomic<bool> failed{false};
        uint64_t mark = 0;      // of the pieces of the ring's first turn, with a sender
        bool by_sender = true;  // where there is one
        explicit Job(std::vector<Piece> p) : pieces(std::move(p)), copied(pieces.size()) {
            for (auto &c : copied) c.store(0);
        }
    };
    // Puts pieces into the ring by a kernel: one launch for up to SENT_MOST of them instead of a copy and an event each.
    struct Sender {
        virtual ~Sender() {}
        // Enqueues pieces from .. to - 1: each to its slot, then its mark behind it.
        virtual hipError_t send(hipStream_t stream, const Mover &m, const Job &j, int from, int to) = 0;
        // hipSuccess while the stream has work left, *over once it has none
        virtual hipError_t ask(hipStream_t stream, bool *over) {
            const hipError_t e = hipStreamQuery(stream);
            *over = e == hipSuccess;
            if (e != hipErrorNotReady) return e;
            (void)hipGetLastError();  // (what a query leaves there is not the error of the next launch)
            return hipSuccess;
        }
        virtual hipError_t lost() = 0;  // the error for pieces that will not come
    };
    char *ring = nullptr;
    uint64_t *marks = nullptr;  // [SENT_SLOTS * MARK_STEP], pinned
    Sender *sender = nullptr;
    uint64_t last_mark = 0;  // (no mark is ever used again)
    hipEvent_t events[SLOTS] = {};
    std::vector<std::thread> workers;
    std::mutex call, mu;  // one transfer at a time; the fields below
    std::condition_variable wake, left;
    Job *job = nullptr;
    uint64_t turn = 0;
    int inside = 0;
    bool stop = false;
    // Destinations of a transfer that is still to come (expect).
    std::vector<Piece> ahead;
    std::vector<std::pair<const char *, const char *>> ahead_ranges;  // what they cover, [from, to)
    std::atomic<int> ahead_next{0};
    bool making = false;              // a helper is at it
    std::atomic<int> ahead_token{0};  // which expect() it is, 0: none
    int tokens = 0;

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
        if (marks) (void)hipHostFree(marks);
        delete sender;
    }
    // helpers: threads beside the caller, who copies as well; fewer, or none, where the system gives no more
    bool start(int helpers) {
        if (!ring && hipHostMalloc((void **)&ring, SLOTS * SLOT, hipHostMallocDefault) != hipSuccess) {
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
    bool sends(const Job &j) const { return sender && j.by_sender; }
    const char *slot_of(const Job &j, int i) const { return sends(j) ? ring + (size_t)(i % SENT_SLOTS) * SENT_SLOT : ring + (size_t)(i % SLOTS) * SLOT; }
    static uint64_t mark_of(const Job &j, int i) { return j.mark + (uint64_t)(i / SENT_SLOTS); }
    bool here(const Job &j, int i) const {
        if (sends(j)) return __atomic_load_n(marks + (size_t)(i % SENT_SLOTS) * MARK_STEP, __ATOMIC_ACQUIRE) == mark_of(j, i);
        return i < j.arrived.load(std::memory_order_acquire);
    }
    void copy(Job &j, int i) {
        memcpy(j.pieces[i].dst, slot_of(j, i), j.pieces[i].bytes);
        j.copied[i].store(1, std::memory_order_release);
        j.done.fetch_add(1, std::memory_order_release);
    }
    // Copies the next piece if it has arrived.
    bool take_arrived(Job &j) {
        int i = j.next.load();
        while (i < (int)j.pieces.size() && here(j, i))
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
            while (!here(j, i)) {
                if (j.failed.load()) return;
                std::this_thread::yield();
            }
            copy(j, i);
        }
    }
    // Has the pages of a piece's destination made, whatever is in them. A caller's memory is often fresh, and threads that copy into the
    // same few megabytes of it wait for each other's page faults; false where the system does not know how.
    static bool make_pages(const Piece &p) {
#ifdef MADV_POPULATE_WRITE
        const uintptr_t page = 4096, a = (uintptr_t)p.dst / page * page, b = ((uintptr_t)p.dst + p.bytes + page - 1) / page * page;
        return madvise((void *)a, b - a, MADV_POPULATE_WRITE) == 0;
#else
        (void)p;
        return false;
#endif
    }
    void wake_workers(Job &j) {
        {
            std::lock_guard<std::mutex> g(mu);
            job = &j;
            turn++;
        }
        wake.notify_all();
    }
    // Whether pages of [dst, dst + bytes) are missing, by a few of them: memory that a caller has used before has them all.
    static bool pages_missing(const char *dst, size_t bytes) {
        const uintptr_t page = 4096, first = (uintptr_t)dst / page, last = ((uintptr_t)dst + bytes - 1) / page;
        for (int i = 0; i <= 4; i++) {
            unsigned char in_core = 1;
            if (mincore((void *)((first + (last - first) * (uintptr_t)i / 4) * page), page, &in_core) == 0 && !(in_core & 1)) return true;
        }
        return false;
    }
    // The pages of these pieces' destinations will be written by a transfer that has not begun: a helper has them made from now on. One:
    // several wait for each other (64 KiB take one thread 6 us, three at once 40).
    // -> what forget() takes, 0 where nothing was begun (no helpers, or another transfer is expected already)
    int expect(std::vector<Piece> pieces) {
        std::lock_guard<std::mutex> g(mu);
        if (ahead_token.load() != 0 || workers.empty() || pieces.empty()) return 0;
        ahead_ranges.clear();
        for (const Piece &p : pieces) {
            if (!ahead_ranges.empty() && ahead_ranges.back().second == p.dst) ahead_ranges.back().second += p.bytes;
            else ahead_ranges.push_back({p.dst, p.dst + p.bytes});
        }
        ahead = std::move(pieces);
        ahead_next.store(0);
        tokens = tokens == 0x7FFFFFFF ? 1 : tokens + 1;
        ahead_token.store(tokens);
        wake.notify_one();
        return tokens;
    }
    // No thread touches what was announced under this token when this returns.
    void forget(int token) {
        std::unique_lock<std::mutex> l(mu);
        if (token == 0 || token != ahead_token.load()) return;
        ahead_next.store((int)ahead.size());
        left.wait(l, [&] { return !making; });
        ahead.clear();
        ahead_token.store(0);
    }
    // Whether a helper makes this piece's pages, or has made them: what is announced is not what every transfer writes, and the
    // helpers may have been busy ever since.
    bool made_ahead(const Piece &p) {
        if (ahead_token.load() == 0) return false;
        std::lock_guard<std::mutex> g(mu);
        if (ahead_token.load() == 0 || (!making && ahead_next.load() == 0)) return false;
        for (const auto &r : ahead_ranges)
            if (r.first <= p.dst && p.dst + p.bytes <= r.second) return true;
        return false;
    }
    bool pages_wanted() const { return !making && ahead_next.load() < (int)ahead.size(); }
    void make_ahead() {
        for (;;) {
            const int i = ahead_next.fetch_add(1);
            if (i >= (int)ahead.size()) return;
            if (!make_pages(ahead[i])) ahead_next.store((int)ahead.size());
        }
    }
    // The threads are out of the job when this returns.
    void finish() {
        std::unique_lock<std::mutex> l(mu);
        job = nullptr;
        left.wait(l, [&] { return inside == 0; });
    }
    // move() with a sender: the caller enqueues up to SENT_MOST pieces whenever their slots are free, and copies what has arrived
    // in between; while nothing has, it makes the destination's pages (those that no helper makes). It never waits for a piece without asking now and then whether the stream still works.
    hipError_t move_sent(hipStream_t stream, Job &j) {
        const int n = (int)j.pieces.size();
        hipError_t err = hipSuccess;
        j.mark = last_mark + 1;
        last_mark += (uint64_t)((n - 1) / SENT_SLOTS) + 1;
        int sent = 0, out = 0, made = 0;  // pieces enqueued; pieces before `out` are out of their slots; pieces whose pages are made
        bool awake = false;
        for (uint32_t polls = 1; j.done.load(std::memory_order_acquire) < n && err == hipSuccess; polls++) {
            while (out < sent && j.copied[out].load(std::memory_order_acquire)) out++;
            if (sent < n) {
                const int to = std::min(n, sent + SENT_MOST);
                if (to - SENT_SLOTS <= out) {
                    err = sender->send(stream, *this, j, sent, to);
                    sent = to;
                    continue;
                }
            }
            if (!awake && here(j, 0)) {  // (the threads sleep through the work that the first piece waits for)
                awake = true;
                wake_workers(j);
            }
            if (awake && take_arrived(j)) continue;  // (not before: piece 256 may take the slot that says that they can be woken)
            made = std::max(made, j.next.load());
            if (made < n) made = made_ahead(j.pieces[made]) || make_pages(j.pieces[made]) ? made + 1 : n;
            else std::this_thread::yield();
            if (polls % 8192 == 0) {  // a stream that has ended without the pieces will not bring them
                bool over = false;
                err = sender->ask(stream, &over);
                for (int i = out; i < sent && over && err == hipSuccess; i++)
                    if (!here(j, i)) err = sender->lost();  // (no slot has been given to a later piece: those wait for `out`)
            }
        }
        if (err != hipSuccess) j.failed.store(true);
        finish();
        return err;
    }
    void work() {
        uint64_t seen = 0;
        std::unique_lock<std::mutex> l(mu);
        for (;;) {
            wake.wait(l, [&] { return stop || (job && turn != seen) || pages_wanted(); });
            if (stop) return;
            if (!(job && turn != seen)) {
                making = true;
                l.unlock();
                make_ahead();
                l.lock();
                making = false;
                left.notify_all();
                continue;
            }
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
        if (sends(j)) return move_sent(stream, j);
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
            if (got == 0) wake_workers(j);  // (the threads sleep through the work that the first piece waits for)
        }
        if (err != hipSuccess) j.failed.store(true);
        else run(j);
        finish();
        return err;
    }
};

}  // namespace vx
