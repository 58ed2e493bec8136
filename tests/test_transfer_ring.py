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
enum { hipSuccess = 0, hipMemcpyDeviceToHost = 2, hipHostMallocDefault = 0, hipEventDisableTiming = 2 };
struct Pending { void *dst; const void *src; size_t bytes; hipEvent_t event; };
static std::deque<Pending> pending;
static hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = malloc(n); return 0; }
static hipError_t hipHostFree(void *p) { free(p); return 0; }
static hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = new int(0); return 0; }
static hipError_t hipEventDestroy(hipEvent_t e) { delete e; return 0; }
static hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, int, hipStream_t) { pending.push_back({d, s, n, nullptr}); return 0; }
static hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { pending.back().event = e; return 0; }
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


# A sender that keeps a launch back until the stream is asked, as a kernel may be late; "lost" leaves the last launch out.
SENDER = HARNESS[:HARNESS.index("int main")] + r"""
#include <atomic>
#include <thread>
struct Late : vx::Mover::Sender {
    std::deque<std::thread> running;
    bool lose = false;
    int sends = 0;
    hipError_t send(hipStream_t, const vx::Mover &m, const vx::Mover::Job &j, int from, int to) override {
        if (to - from < 1 || to - from > vx::Mover::SENT_MOST) return 5;
        sends++;
        if (lose && to == (int)j.pieces.size()) return 0;
        if (!running.empty()) running.back().join(), running.pop_back();  // (one launch behind the other)
        running.emplace_back([&m, &j, from, to] {
            for (int i = from; i < to; i++) {
                std::this_thread::yield();
                if (i >= vx::Mover::SENT_SLOTS && !j.copied[i - vx::Mover::SENT_SLOTS].load()) abort();  // the slot is still in use
                memcpy(m.ring + (size_t)(i % vx::Mover::SENT_SLOTS) * vx::Mover::SENT_SLOT, j.pieces[i].src, j.pieces[i].bytes);
                __atomic_store_n(m.marks + (size_t)(i % vx::Mover::SENT_SLOTS) * vx::Mover::MARK_STEP, vx::Mover::mark_of(j, i), __ATOMIC_RELEASE);
            }
        });
        return 0;
    }
    void wait() { while (!running.empty()) running.back().join(), running.pop_back(); }
    hipError_t ask(hipStream_t, bool *over) override { *over = lose; return 0; }
    hipError_t lost() override { return 9; }
};
int main(int argc, char **argv) {
    const int helpers = atoi(argv[1]);
    vx::Mover m;
    m.marks = (uint64_t *)calloc(vx::Mover::SENT_SLOTS * vx::Mover::MARK_STEP, 8);
    Late *late = new Late;
    m.sender = late;
    if (!m.start(helpers) || (int)m.workers.size() != helpers) return 2;
    const size_t piece = 4099;
    for (int i = 2; i < argc; i++) {
        const int n = abs(atoi(argv[i]));
        late->lose = atoi(argv[i]) < 0;
        std::string from(n * piece, 0), to(n * piece, 0);
        for (size_t k = 0; k < from.size(); k++) from[k] = (char)(k * 2654435761u >> 13);
        std::vector<vx::Mover::Piece> pieces;
        for (int k = 0; k < n; k++) pieces.push_back({&to[k * piece], &from[k * piece], piece});
        vx::Mover::Job job(std::move(pieces));
        const int rc = m.move(0, job);
        late->wait();
        if (late->lose ? rc != 9 : rc != 0 || from != to) return 3;
        printf("%d ok\n", atoi(argv[i]));
        fflush(stdout);
    }
    return 0;
}
"""


@pytest.mark.parametrize("helpers", [0, 1, 6])
def test_every_sent_piece_arrives(tmp_path, helpers):
    """Both sides of a launch (64 pieces), of the ring (256 slots) and of several turns of it; a stream that ends without its
    last launch is an error and not a wait without an end, and what comes after it is whole again."""
    src, exe = tmp_path / "sent.cpp", tmp_path / "sent"
    src.write_text(SENDER)
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I" + os.path.join(ROOT, "vexel_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    sizes = [1, 63, 64, 65, 255, 256, 257, -3, 320, 321, -300, 1000]
    r = subprocess.run([str(exe), str(helpers)] + [str(n) for n in sizes], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.split("\n")[:-1] == ["%d ok" % n for n in sizes], (r.returncode, r.stdout)
