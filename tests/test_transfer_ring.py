"""The ring of large downloads (csrc/transfer_ring.h) against copies made on the host: every number of helper threads, none
among them, at both sides of the ring's sixteen pieces and over several turns of it."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# A copy happens when an event behind it is waited for, as late as the ring may expect it.
HARNESS = r"""
#include <stdio.h>
#include <stdlib.h>
#include <deque>
#include <string>
typedef int hipError_t;
typedef int hipStream_t;
typedef int *hipEvent_t;
enum { hipSuccess = 0, hipErrorNotReady = 600, hipMemcpyDeviceToHost = 2, hipHostMallocDefault = 0, hipEventDisableTiming = 2 };
struct Pending { void *dst; const void *src; size_t bytes; hipEvent_t event; };
static std::deque<Pending> pending;
static hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = malloc(n); return 0; }
static hipError_t hipHostFree(void *p) { free(p); return 0; }
static hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = new int(0); return 0; }
static hipError_t hipEventDestroy(hipEvent_t e) { delete e; return 0; }
static hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, int, hipStream_t) { pending.push_back({d, s, n, nullptr}); return 0; }
static hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { pending.back().event = e; return 0; }
static hipError_t last_error = hipSuccess;
static hipError_t hipGetLastError() { const hipError_t e = last_error; last_error = hipSuccess; return e; }
static hipError_t hipStreamQuery(hipStream_t);
#include <string.h>
static hipError_t hipEventSynchronize(hipEvent_t e) {
    while (!pending.empty()) {
        Pending p = pending.front();
        pending.pop_front();
        memcpy(p.dst, p.src, p.bytes);
        if (p.event == e) break;
    }
    return 0;
}
#include "transfer_ring.h"
static hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
int main(int argc, char **argv) {
    const int helpers = atoi(argv[1]);
    vx::Mover m;
    if (!m.start(helpers) || (int)m.workers.size() != helpers) return 2;
    const size_t piece = 4099;
    for (int i = 2; i < argc; i++) {
        const int n = atoi(argv[i]);
        std::string from(n * piece, 0), to(n * piece, 0);
        for (size_t k = 0; k < from.size(); k++) from[k] = (char)(k * 2654435761u >> 13);
        std::vector<vx::Mover::Piece> pieces;
        for (int k = 0; k < n; k++) pieces.push_back({&to[k * piece], &from[k * piece], piece});
        vx::Mover::Job job(std::move(pieces));
        if (m.move(0, job) != 0 || from != to) return 3;
        printf("%d ok\n", n);
        fflush(stdout);
    }
    return 0;
}
"""


@pytest.fixture(scope="module")
def ring(tmp_path_factory):
    at = tmp_path_factory.mktemp("ring")
    src, exe = at / "ring.cpp", at / "ring"
    src.write_text(HARNESS)
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I" + os.path.join(ROOT, "vexel_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    return str(exe)


@pytest.mark.parametrize("helpers", [0, 1, 2, 6])
def test_every_piece_arrives(ring, helpers):
    sizes = [1, 15, 16, 17, 32, 40, 41, 200]
    r = subprocess.run([ring, str(helpers)] + [str(n) for n in sizes], capture_output=True, text=True, timeout=30)
    assert r.returncode == 0 and r.stdout.split("\n")[:-1] == ["%d ok" % n for n in sizes], (r.returncode, r.stdout)


# A sender whose launches run one behind the other on a thread, as on a stream. "h": they begin when the stream is asked about, as behind a
# long step; "s": a helper thread copies its first piece when the stream has been found at its end; "l": the last launch is lost.
SENDER = HARNESS[:HARNESS.index('#include "transfer_ring.h"')] + r"""
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <mutex>
#include <thread>
static std::thread::id caller;
static std::atomic<bool> slow{false};
static std::atomic<int> holding{0}, found_over{0};
static void await(const std::atomic<int> &what) {
    for (const auto end = std::chrono::steady_clock::now() + std::chrono::seconds(20); what.load() == 0; std::this_thread::yield())
        if (std::chrono::steady_clock::now() > end) abort();
}
static thread_local bool device = false;
static void copy_slowly(void *d, const void *s, size_t n) {
    if (slow.load() && !device) {
        if (std::this_thread::get_id() == caller) await(holding);  // (so that the helpers get pieces)
        else holding++, await(found_over);
    }
    memcpy(d, s, n);
}
#define memcpy copy_slowly
#include "transfer_ring.h"
struct Late : vx::Mover::Sender {
    struct Launch { const vx::Mover *m; const vx::Mover::Job *j; int from, to; };
    std::mutex mu;
    std::condition_variable more;
    std::deque<Launch> queue;
    int free_to_run = 0, launched = 0, finished = 0;
    bool hold = false, lose = false, stop = false;
    std::thread runs{[this] { run(); }};
    ~Late() override {
        { std::lock_guard<std::mutex> g(mu); stop = true; }
        more.notify_all();
        runs.join();
    }
    void run() {
        device = true;
        std::unique_lock<std::mutex> l(mu);
        for (;;) {
            more.wait(l, [&] { return stop || (finished < launched && (!hold || finished < free_to_run)); });
            if (stop) return;
            const Launch a = queue.front();
            l.unlock();
            for (int i = a.from; i < a.to; i++) {
                std::this_thread::yield();
                if (i >= vx::Mover::SENT_SLOTS && !a.j->copied[i - vx::Mover::SENT_SLOTS].load()) abort();  // the slot is still in use
                memcpy(a.m->ring + (size_t)(i % vx::Mover::SENT_SLOTS) * vx::Mover::SENT_SLOT, a.j->pieces[i].src, a.j->pieces[i].bytes);
                __atomic_store_n(a.m->marks + (size_t)(i % vx::Mover::SENT_SLOTS) * vx::Mover::MARK_STEP, vx::Mover::mark_of(*a.j, i), __ATOMIC_RELEASE);
            }
            l.lock();
            queue.pop_front();
            finished++;
        }
    }
    hipError_t send(hipStream_t, const vx::Mover &m, const vx::Mover::Job &j, int from, int to) override {
        if (to - from < 1 || to - from > vx::Mover::SENT_MOST) return 5;
        if (lose && to == (int)j.pieces.size()) return 0;
        { std::lock_guard<std::mutex> g(mu); queue.push_back({&m, &j, from, to}); launched++; }
        more.notify_all();
        return hipGetLastError();
    }
    hipError_t query() {
        std::lock_guard<std::mutex> g(mu);
        free_to_run = launched;
        more.notify_all();
        if (finished == launched) found_over++;
        return finished == launched ? hipSuccess : hipErrorNotReady;
    }
    hipError_t lost() override { return 9; }
};
static Late *late = nullptr;
static hipError_t hipStreamQuery(hipStream_t) {  // a runtime that keeps "not ready" as the last error
    const hipError_t e = late->query();
    return e == hipSuccess ? e : last_error = e;
}
int main(int argc, char **argv) {
    const int helpers = atoi(argv[1]);
    caller = std::this_thread::get_id();
    vx::Mover m;
    m.marks = (uint64_t *)calloc(vx::Mover::SENT_SLOTS * vx::Mover::MARK_STEP, 8);
    m.sender = late = new Late;
    if (!m.start(helpers) || (int)m.workers.size() != helpers) return 2;
    const size_t piece = 4099;
    for (int i = 2; i < argc; i++) {
        const int n = atoi(argv[i] + strcspn(argv[i], "0123456789"));
        { std::lock_guard<std::mutex> g(late->mu); late->hold = strchr(argv[i], 'h'), late->lose = strchr(argv[i], 'l'); }
        slow = strchr(argv[i], 's') && helpers > 0;
        holding = 0, found_over = 0;
        std::string from(n * piece, 0), to(n * piece, 0);
        for (size_t k = 0; k < from.size(); k++) from[k] = (char)(k * 2654435761u >> 13);
        std::vector<vx::Mover::Piece> pieces;
        for (int k = 0; k < n; k++) pieces.push_back({&to[k * piece], &from[k * piece], piece});
        vx::Mover::Job job(std::move(pieces));
        const int rc = m.move(0, job);
        if (late->lose ? rc != 9 : rc != 0 || from != to) return 3;
        if (slow && (holding.load() == 0 || found_over.load() == 0)) return 4;
        if (late->hold && late->free_to_run == 0) return 6;
        printf("%s ok\n", argv[i]);
        fflush(stdout);
    }
    return 0;
}
"""


@pytest.mark.parametrize("helpers", [0, 1, 6])
def test_every_sent_piece_arrives(tmp_path, helpers):
    """Both sides of a launch (64 pieces), of the ring (256 slots) and of several turns of it; launches that come late; a stream found
    at its end while pieces that have arrived are still to be copied, which is no loss; a stream that ends without its last launch,
    which is an error and not a wait without an end, and what comes after it is whole again."""
    src, exe = tmp_path / "sent.cpp", tmp_path / "sent"
    src.write_text(SENDER)
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I" + os.path.join(ROOT, "vexel_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    jobs = ["1", "63", "64", "65", "255", "256", "257", "l3", "320", "321", "l300", "1000", "h1", "h257", "h600", "s65", "s257", "s320", "s600", "hs400", "l65", "s256"]
    r = subprocess.run([str(exe), str(helpers)] + jobs, capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.split("\n")[:-1] == [j + " ok" for j in jobs], (r.returncode, r.stdout)


# Memory that is announced before its transfer: all its pages come, what is in it stays, nothing touches it once it is forgotten.
AHEAD = HARNESS[:HARNESS.index("int main(")] + r"""
#include <chrono>
static const size_t PAGE = 4096, N = 600 * PAGE + 123;
static char *fresh() { return (char *)mmap(nullptr, N, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0); }
static int missing(const char *p) {
    int n = 0;
    for (size_t i = 0; i * PAGE < N; i++) {
        unsigned char c = 0;
        if (mincore((void *)(p + i * PAGE), PAGE, &c) != 0 || !(c & 1)) n++;
    }
    return n;
}
static std::vector<vx::Mover::Piece> pieces_of(char *dst, const char *src) {
    std::vector<vx::Mover::Piece> p;
    for (size_t at = 0; at < N; at += vx::Mover::SENT_SLOT) p.push_back({dst + at, src ? src + at : nullptr, std::min(vx::Mover::SENT_SLOT, N - at)});
    return p;
}
int main(int argc, char **argv) {
    const int helpers = atoi(argv[1]);
    vx::Mover m;
    if (!m.start(helpers)) return 2;
    char *a = fresh();
    a[5 * PAGE + 7] = 42;
    if (!vx::Mover::pages_missing(a, N)) return 3;
    const int t = m.expect(pieces_of(a, nullptr));
    if ((t != 0) != (helpers > 0)) return 4;
    if (helpers > 0 && m.expect(pieces_of(a, nullptr)) != 0) return 5;  // one at a time
    m.forget(t + 1);                                                    // (somebody else's)
    const auto end = std::chrono::steady_clock::now() + std::chrono::seconds(20);
    while (helpers > 0 && missing(a) > 0)
        if (std::chrono::steady_clock::now() > end) return 6;
    std::string from(N, 0);
    for (size_t k = 0; k < N; k++) from[k] = (char)(k * 2654435761u >> 13);
    if (helpers > 0 && (a[5 * PAGE + 7] != 42 || a[5 * PAGE + 8] != 0 || vx::Mover::pages_missing(a, N))) return 7;
    vx::Mover::Job job(pieces_of(a, from.data()));
    if (m.move(0, job) != 0 || memcmp(a, from.data(), N) != 0) return 8;  // while it is still announced
    m.forget(t);
    m.forget(t);
    munmap(a, N);
    for (int i = 0; i < 200; i++) {  // forgotten at once, with and without the transfer, and gone afterwards
        char *b = fresh();
        const int u = m.expect(pieces_of(b, nullptr));
        if ((u != 0) != (helpers > 0) || (u != 0 && u == t)) return 9;
        if (i % 3 == 0) {
            vx::Mover::Job again(pieces_of(b, from.data()));
            if (m.move(0, again) != 0 || memcmp(b, from.data(), N) != 0) return 10;
        }
        m.forget(u);
        munmap(b, N);
    }
    char *gone = fresh();  // memory that is not there is nobody's fault
    munmap(gone, N);
    m.forget(m.expect(pieces_of(gone, nullptr)));
    puts("ok");
    return 0;
}
"""


@pytest.mark.parametrize("helpers", [0, 1, 6])
def test_pages_of_expected_transfers(tmp_path, helpers):
    src, exe = tmp_path / "ahead.cpp", tmp_path / "ahead"
    src.write_text(AHEAD)
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I" + os.path.join(ROOT, "vexel_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe), str(helpers)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout)


# Which pages the caller of a transfer makes itself while another destination, its own, or a part of its own is announced.
BESIDE = SENDER[:SENDER.index("int main(")].replace("#define memcpy copy_slowly", r"""#include <sys/mman.h>
static char *made_from = nullptr;
static size_t made_bytes = 0;
static int noted_madvise(void *a, size_t n, int what) {  // (of the caller's, one after the other)
    if (std::this_thread::get_id() == caller) {
        if (!made_from) made_from = (char *)a;
        made_bytes += n;
    }
    return madvise(a, n, what);
}
#define madvise noted_madvise
#define memcpy copy_slowly""") + r"""
static const size_t SLOT = vx::Mover::SENT_SLOT, N = 10 * SLOT;
static char *fresh() { return (char *)mmap(nullptr, N, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0); }
static void add(std::vector<vx::Mover::Piece> &to, char *dst, const char *src) {
    for (size_t at = 0; at < N; at += SLOT) to.push_back({dst + at, src ? src + at : nullptr, SLOT});
}
static bool missing(const char *p) {
    unsigned char in_core[N / 4096];
    if (mincore((void *)p, N, in_core) != 0) return true;
    for (unsigned char c : in_core)
        if (!(c & 1)) return true;
    return false;
}
int main(int argc, char **argv) {
    caller = std::this_thread::get_id();
    vx::Mover m;
    m.marks = (uint64_t *)calloc(vx::Mover::SENT_SLOTS * vx::Mover::MARK_STEP, 8);
    m.sender = late = new Late;
    late->hold = true;  // (the first piece comes when all pages that the caller makes have been made)
    if (!m.start(atoi(argv[1]))) return 2;
    std::string from(N, 0);
    for (size_t k = 0; k < N; k++) from[k] = (char)(k * 2654435761u >> 13);
    for (const char *what : {"other", "own", "part"}) {
        char *x = fresh(), *y = fresh();
        std::vector<vx::Mover::Piece> announced, pieces;
        add(announced, what[1] == 'w' ? x : y, nullptr);
        const int token = m.expect(announced);
        if (token == 0) return 3;
        for (const auto end = std::chrono::steady_clock::now() + std::chrono::seconds(20); missing(announced[0].dst); std::this_thread::yield())
            if (std::chrono::steady_clock::now() > end) return 4;
        if (what[0] == 'p') add(pieces, y, from.data());
        add(pieces, x, from.data());
        made_from = nullptr, made_bytes = 0;
        vx::Mover::Job job(pieces);
        if (m.move(0, job) != 0 || memcmp(x, from.data(), N) != 0) return 5;
        if (what[0] == 'p' && memcmp(y, from.data(), N) != 0) return 6;
        if (what[1] == 'w' ? made_bytes != 0 : made_from != x || made_bytes != N) return 7;
        m.forget(token);
        munmap(x, N);
        munmap(y, N);
        printf("%s ok\n", what);
    }
    return 0;
}
"""


@pytest.mark.parametrize("helpers", [1, 6])
def test_pages_beside_an_announcement(tmp_path, helpers):
    src, exe = tmp_path / "beside.cpp", tmp_path / "beside"
    src.write_text(BESIDE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I" + os.path.join(ROOT, "vexel_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe), str(helpers)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "other ok\nown ok\npart ok\n", (r.returncode, r.stdout)
