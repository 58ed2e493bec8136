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
