// Copies between host and device memory. C ABI: include/vexel_hip.h.
//
// A step of a model gives its caller megabytes of logits in ordinary (pageable) memory, often memory that has just been
// allocated and is not there yet. The runtime's own copy of that kind moves a piece at a time through a buffer of its own and
// copies (and takes the page faults of) each on the calling thread: 32 MiB take 3.4 ms where the bus needs 0.6 ms.
// Here the pieces go through a ring of pinned memory one behind the other, and a few threads of the backend copy
// those that have arrived while later ones are on their way. Small uploads go through pinned memory without waiting.
//
// What bounds a download is the bus (56 GB/s), and between its pieces it stood still: a copy of the runtime's with an event
// behind it costs 13 us beside the bytes, so 4.1 MB in eight pieces took 206 us of 73 and 32.8 MB in 32 pieces 1047 of 586. One
// kernel sends up to 64 pieces of 64 KiB instead, each with a mark in pinned memory behind it that the threads look at:
// 4.1 MB in 95 us, 32.8 MB in 633, 1 MB in 44 (88 before). More threads than six, none.
#include <memory>

#include "common.h"
#include "transfer_ring.h"

namespace vx {

void mover_destroy(Mover *m) { delete m; }

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// n bytes by the threads of a workgroup, in pieces of what both addresses are aligned to
__device__ __forceinline__ void copy_bytes(char *dst, const char *src, uint32_t n, int tid, int threads) {
    const uintptr_t at = (uintptr_t)dst | (uintptr_t)src;
    uint32_t done = 0;
    if ((at & 15) == 0) {
        for (uint32_t k = tid; k < n / 16; k += threads) ((u32x4 *)dst)[k] = ((const u32x4 *)src)[k];
        done = n / 16 * 16;
    } else if ((at & 3) == 0) {
        for (uint32_t k = tid; k < n / 4; k += threads) ((uint32_t *)dst)[k] = ((const uint32_t *)src)[k];
        done = n / 4 * 4;
    } else if (((uintptr_t)dst & 3) == 0) {  // (the two words that hold a word's bytes; of memory that begins and ends on words)
        const uint32_t *words = (const uint32_t *)((uintptr_t)src & ~(uintptr_t)3), off = (uintptr_t)src & 3;
        for (uint32_t k = tid; k < n / 4; k += threads) ((uint32_t *)dst)[k] = __builtin_amdgcn_alignbyte(words[k + 1], words[k], off);
        done = n / 4 * 4;
    }
    for (uint32_t k = done + tid; k < n; k += threads) dst[k] = src[k];
}

struct SendArgs {
    const char *src[Mover::SENT_MOST];
    uint32_t bytes[Mover::SENT_MOST];
    char *ring;
    uint64_t *marks;
    uint64_t mark;
    int from, count;
};
// Pieces from .. from + count - 1 of a job to their slots of the ring, a workgroup a piece at a time; then the piece's mark. The
// few workgroups take the pieces in order, so that the first ones are there long before the last (16 of them: 4.1 MB in 95 us, 32
// in 100, 64 in 123). All loads of a piece are asked for before the first store: 16 of 16 bytes a thread.
constexpr int SEND_GROUPS = 16, SEND_THREADS = 256, SEND_VECS = (int)(Mover::SENT_SLOT / 16 / SEND_THREADS);
__global__ void __launch_bounds__(SEND_THREADS) send_kernel(const SendArgs a) {
    const int tid = threadIdx.x;
    for (int p = blockIdx.x; p < a.count; p += gridDim.x) {
        const int i = a.from + p, slot = i % Mover::SENT_SLOTS;
        const char *src = a.src[p];
        char *dst = a.ring + (size_t)slot * Mover::SENT_SLOT;
        const uint32_t n = a.bytes[p];
        if (n == Mover::SENT_SLOT && ((uintptr_t)src & 15) == 0) {
            const u32x4 *s4 = (const u32x4 *)src;
            u32x4 v[SEND_VECS];
#pragma unroll
            for (int k = 0; k < SEND_VECS; k++) v[k] = s4[tid + k * SEND_THREADS];
#pragma unroll
            for (int k = 0; k < SEND_VECS; k++) ((u32x4 *)dst)[tid + k * SEND_THREADS] = v[k];
        } else {
            copy_bytes(dst, src, n, tid, SEND_THREADS);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");  // (system scope: each thread's bytes are there before any thread is past the barrier)
        __syncthreads();
        if (tid == 0)
            __hip_atomic_store(a.marks + (size_t)slot * Mover::MARK_STEP, a.mark + (uint64_t)(i / Mover::SENT_SLOTS), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// Small uploads that lie in pinned memory one behind the other, a workgroup each.
constexpr int SCATTER_MOST = 64;
struct ScatterArgs {
    const char *from;
    char *dst[SCATTER_MOST];
    uint32_t at[SCATTER_MOST], bytes[SCATTER_MOST];
};
__global__ void __launch_bounds__(SEND_THREADS) scatter_kernel(const ScatterArgs a) {
    const int i = blockIdx.x;
    copy_bytes(a.dst[i], a.from + a.at[i], a.bytes[i], threadIdx.x, SEND_THREADS);
}

namespace {
struct KernelSender : Mover::Sender {
    hipError_t send(hipStream_t stream, const Mover &m, const Mover::Job &j, int from, int to) override {
        SendArgs a = {};
        for (int i = from; i < to; i++) a.src[i - from] = j.pieces[i].src, a.bytes[i - from] = (uint32_t)j.pieces[i].bytes;
        a.ring = m.ring, a.marks = m.marks, a.mark = j.mark, a.from = from, a.count = to - from;
        send_kernel<<<std::min(SEND_GROUPS, to - from), SEND_THREADS, 0, stream>>>(a);
        return hipGetLastError();
    }
    hipError_t lost() override { return hipErrorUnknown; }
};

}  // namespace

// (The runtime's copy says what is wrong with other memory.)
bool device_memory(const vx_backend *be, const void *src, size_t bytes) {
    hipPointerAttribute_t a;
    hipDeviceptr_t base = nullptr;
    size_t size = 0;
    const bool ok = hipPointerGetAttributes(&a, src) == hipSuccess && a.type == hipMemoryTypeDevice && a.device == be->device &&
                    hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)src) == hipSuccess &&
                    (size_t)((const char *)src - (const char *)base) + bytes <= size;
    if (!ok) (void)hipGetLastError();
    return ok;
}

namespace {
// Coherent pinned memory for the ring and its marks: what a kernel has written there is seen by the host while the kernel runs.
// Without it the runtime's copies fill the ring.
void use_sender(Mover *m) {
    const size_t marks = Mover::SENT_SLOTS * Mover::MARK_STEP * sizeof(uint64_t);
    if (hipHostMalloc((void **)&m->ring, Mover::SLOTS * Mover::SLOT, hipHostMallocCoherent) != hipSuccess) m->ring = nullptr;
    if (m->ring && hipHostMalloc((void **)&m->marks, marks, hipHostMallocCoherent) != hipSuccess) m->marks = nullptr;
    if (m->ring && m->marks) {
        memset(m->marks, 0, marks);
        m->sender = new KernelSender();
        return;
    }
    if (m->ring) (void)hipHostFree(m->ring);
    m->ring = nullptr;
    (void)hipGetLastError();
}
}  // namespace

// The backend's pinned megabyte: a word of vx_argmax's, small downloads' marks, staged uploads, small downloads.
constexpr size_t NOTES_AT = 32 << 10, UP_AT = 64 << 10, UP_BYTES = 448 << 10, DOWN_AT = 512 << 10, DOWN_BYTES = 512 << 10, UP_MOST = 64 << 10;

// The backend's ring and threads, made by the first large download; null where they could not be made.
static Mover *mover_of(vx_backend *be) {
    std::lock_guard<std::mutex> g(be->stage_mu);
    if (!be->mover) {  // (kept when it is whole, whatever throws before)
        std::unique_ptr<Mover> made(new Mover());
        use_sender(made.get());
        if (made->start(std::min<int>(Mover::MAX_WORKERS, std::max(1u, std::thread::hardware_concurrency()) - 1)))
            be->mover = made.release();
        else
            (void)hipGetLastError();
    }
    return be->mover;
}

// A small download. The runtime's takes a copy of its own for every range, and its wait for the stream comes back 15 - 20 us late behind more than six
// launches. One launch of send_kernel instead, into the pinned megabyte's slots, and the caller looks at its marks, which keeps its core busy as the
// runtime's wait does (either takes as much processor time as it lasts, behind 5 us of work and behind 13 ms): 4
// bytes behind 0, 1, 6, 8 and 20 short kernels 12.7, 15.8, 30, 62 and 106 us -> 8.9, 12, 27, 33 and 68, 128 KB behind 1, 8 and 20 of them 27, 65 and
// 105 -> 17, 38 and 74, all eight slots of 64 KiB 40, 102 -> 38, 96 behind 1 and 20.
// The runtime's is the sooner one where nothing is ahead and one range comes that is long for a workgroup a slot (64, 128 and 512 KiB 12.3, 15.0 and 30.1 us
// against 16.8, 18.6 and 33.7; 16 KiB 14.3 and 14.1; from an address that is no multiple of 16, by words, 16 KiB 14.2 and 15.3, 64 KiB 12.4 and 22.8). Whether
// something is ahead is not asked of the stream: the question costs it 12 us.
// VX_ERR_UNSUPPORTED, with nothing done, for such a one, where a range is nothing that a kernel can read, and where the ranges need more slots.
static int download_noted(vx_backend *be, int n, void *const *dst, const void *const *src, const size_t *bytes) {
    constexpr int SLOTS = (int)(DOWN_BYTES / Mover::SENT_SLOT);
    constexpr size_t LONG = 16 << 10, LONG_APART = 4 << 10;
    int ranges = 0;
    size_t slots = 0;
    bool is_long = false;
    for (int i = 0; i < n; i++) {
        if (!src[i] || bytes[i] == 0) continue;
        ranges++, slots += (bytes[i] + Mover::SENT_SLOT - 1) / Mover::SENT_SLOT;
        is_long = is_long || bytes[i] > ((uintptr_t)src[i] % 16 == 0 ? LONG : LONG_APART);
    }
    if (slots > SLOTS || (ranges == 1 && is_long && be->at_rest.load(std::memory_order_relaxed))) return VX_ERR_UNSUPPORTED;
    SendArgs a = {};
    char *to[SLOTS];
    for (int i = 0; i < n; i++) {
        if (!src[i] || bytes[i] == 0) continue;
        if (!device_memory(be, src[i], bytes[i])) return VX_ERR_UNSUPPORTED;
        for (size_t at = 0; at < bytes[i]; at += Mover::SENT_SLOT, a.count++) {
            a.src[a.count] = (const char *)src[i] + at, a.bytes[a.count] = (uint32_t)std::min(Mover::SENT_SLOT, bytes[i] - at);
            to[a.count] = (char *)dst[i] + at;
        }
    }
    char *stage = (char *)be->host_stage;
    a.ring = stage + DOWN_AT, a.marks = (uint64_t *)(stage + NOTES_AT), a.mark = ++be->note_mark;
    send_kernel<<<a.count, SEND_THREADS, 0, be->stream>>>(a);
    VX_CHECK_LAUNCH();
    KernelSender stream_state;
    for (int i = 0; i < a.count; i++) {
        const auto here = [&] { return __atomic_load_n(a.marks + (size_t)i * Mover::MARK_STEP, __ATOMIC_ACQUIRE) == a.mark; };
        for (uint32_t polls = 1; !here(); polls++) {
            std::this_thread::yield();
            if (polls % 8192 != 0) continue;  // a stream that has ended without the mark will not bring it
            bool over = false;
            VX_CHECK_HIP(stream_state.ask(be->stream, &over));
            if (over && !here()) VX_CHECK_HIP(stream_state.lost());
        }
        memcpy(to[i], a.ring + (size_t)i * Mover::SENT_SLOT, a.bytes[i]);
    }
    return VX_OK;
}

static int download(vx_backend *be, int n, void *const *dst, const void *const *src, const size_t *bytes) {
    size_t total = 0;
    for (int i = 0; i < n; i++)
        if (src[i]) total += (bytes[i] + 63) / 64 * 64;
    if (total == 0) return VX_OK;
    for (int i = 0; i < n; i++) VX_REQUIRE(!src[i] || bytes[i] == 0 || dst[i] != nullptr, "vx_to_host: null destination");
    if (total <= DOWN_BYTES) {
        std::lock_guard<std::mutex> g(be->stage_mu);
        const int rc = download_noted(be, n, dst, src, bytes);
        if (rc != VX_ERR_UNSUPPORTED) return rc;
        char *stage = (char *)be->host_stage + DOWN_AT;
        size_t at = 0;
        for (int i = 0; i < n; i++) {
            if (!src[i] || bytes[i] == 0) continue;
            VX_CHECK_HIP(hipMemcpyAsync(stage + at, src[i], bytes[i], hipMemcpyDeviceToHost, be->stream));
            at += (bytes[i] + 63) / 64 * 64;
        }
        VX_CHECK_HIP(hipStreamSynchronize(be->stream));
        at = 0;
        for (int i = 0; i < n; i++) {
            if (!src[i] || bytes[i] == 0) continue;
            memcpy(dst[i], stage + at, bytes[i]);
            at += (bytes[i] + 63) / 64 * 64;
        }
        return VX_OK;
    }
    bool pinned = false;  // (memory that the device reaches by itself needs no ring)
    for (int i = 0; i < n; i++) {
        hipPointerAttribute_t a;
        if (src[i] && bytes[i] > 0 && hipPointerGetAttributes(&a, dst[i]) == hipSuccess) pinned = pinned || a.type != hipMemoryTypeUnregistered;
        else (void)hipGetLastError();
    }
    Mover *mover = pinned ? nullptr : mover_of(be);
    if (!mover) {
        for (int i = 0; i < n; i++)
            if (src[i] && bytes[i] > 0) VX_CHECK_HIP(hipMemcpyAsync(dst[i], src[i], bytes[i], hipMemcpyDeviceToHost, be->stream));
        VX_CHECK_HIP(hipStreamSynchronize(be->stream));
        return VX_OK;
    }
    // pieces of a slot; of the runtime's larger slots an eighth, so that the threads have something to share, of 256 KiB up
    bool by_sender = mover->sender != nullptr;
    for (int i = 0; i < n && by_sender; i++) by_sender = !src[i] || bytes[i] == 0 || device_memory(be, src[i], bytes[i]);
    const size_t most = by_sender ? Mover::SENT_SLOT : std::min(Mover::SLOT, std::max((size_t)256 << 10, total / 8 / 4096 * 4096));
    std::vector<Mover::Piece> pieces;
    for (int i = 0; i < n; i++) {
        if (!src[i]) continue;
        for (size_t at = 0; at < bytes[i]; at += most)
            pieces.push_back({(char *)dst[i] + at, (const char *)src[i] + at, std::min(most, bytes[i] - at)});
    }
    std::lock_guard<std::mutex> g(mover->call);
    Mover::Job job(std::move(pieces));
    job.by_sender = by_sender;
    VX_CHECK_HIP(mover->move(be->stream, job));
    return VX_OK;
}

int stage_upload(vx_backend *be, const void *src_host, size_t bytes, const char **at) {
    const size_t room = (bytes + 63) / 64 * 64;
    VX_REQUIRE(bytes <= UP_MOST, "staged upload of %zu bytes", bytes);
    if (be->stage_used + room > UP_BYTES) {
        VX_CHECK_HIP(hipStreamSynchronize(be->stream));
        be->stage_used = 0;
    }
    char *to = (char *)be->host_stage + UP_AT + be->stage_used;
    be->stage_used += room;
    memcpy(to, src_host, bytes);
    *at = to;
    return VX_OK;
}

}  // namespace vx

using namespace vx;

extern "C" {

int vx_to_host_many(vx_backend *be, int n, void *const *dst_host, const void *const *src, const size_t *bytes) {
    int rc = enter_to_wait(be);
    if (rc) return rc;
    if (n == 0) return VX_OK;
    VX_REQUIRE(n > 0 && dst_host && src && bytes, "vx_to_host: bad arguments");
    VX_REQUIRE(!be->capturing, "vx_to_host during graph capture");
    bool any = false;
    for (int i = 0; i < n; i++) any = any || (src[i] && bytes[i] > 0);
    try {
        rc = download(be, n, dst_host, src, bytes);
    } catch (...) {
        set_error("vx_to_host: out of host memory");
        return VX_ERR_OOM;
    }
    if (rc == VX_OK && any) be->at_rest.store(true, std::memory_order_relaxed);
    return rc;
}

// What bounds a short step whose caller wants large logits in memory that is not there yet is the page faults: 4.1 MB of them take
// one thread 500 us, the download began with them only once the whole step was enqueued, and what had arrived by then waited for its pages
// (32 sequences of a bfloat16 model of four layers: 270 - 420 us from the first piece to the last, 75 now; 695 -> 610 us a step, and the same as
// before, 590 - 600, in memory that is there). Below 2 MiB the pages are made in the time that the device takes after the last launch.
constexpr size_t EXPECT_LEAST = (size_t)2 << 20;
int vx_to_host_expect(vx_backend *be, int n, void *const *dst_host, const size_t *bytes, int *token) {
    int rc = enter(be);
    if (rc) return rc;
    VX_REQUIRE(n >= 0 && (n == 0 || (dst_host && bytes)) && token, "vx_to_host_expect: bad arguments");
    *token = 0;
    size_t total = 0;
    for (int i = 0; i < n; i++)
        if (dst_host[i]) total += (bytes[i] + 63) / 64 * 64;
    if (total < EXPECT_LEAST || be->capturing) return VX_OK;
    try {
        std::vector<Mover::Piece> pieces;
        for (int i = 0; i < n; i++) {
            if (!dst_host[i] || bytes[i] == 0 || !Mover::pages_missing((const char *)dst_host[i], bytes[i])) continue;
            for (size_t at = 0; at < bytes[i]; at += Mover::SENT_SLOT)
                pieces.push_back({(char *)dst_host[i] + at, nullptr, std::min(Mover::SENT_SLOT, bytes[i] - at)});
        }
        if (Mover *m = pieces.empty() ? nullptr : mover_of(be)) *token = m->expect(std::move(pieces));
    } catch (...) {  // (a hint: the download itself says what is wrong)
    }
    return VX_OK;
}

void vx_to_host_forget(vx_backend *be, int token) {
    if (be && token && be->mover) be->mover->forget(token);
}

int vx_to_host(vx_backend *be, void *dst_host, const void *src, size_t bytes) {
    int rc = enter_to_wait(be);
    if (rc) return rc;
    if (!src || bytes == 0) return VX_OK;
    return vx_to_host_many(be, 1, &dst_host, &src, &bytes);
}

int vx_to_device_staged(vx_backend *be, void *dst, const void *src_host, size_t bytes) {
    if (bytes > UP_MOST) return vx_to_device(be, dst, src_host, bytes);
    int rc = enter(be);
    if (rc) return rc;
    if (!dst || bytes == 0) return VX_OK;
    VX_REQUIRE(src_host != nullptr, "vx_to_device_staged: null source");
    VX_REQUIRE(!be->capturing, "vx_to_device_staged during graph capture");
    items_written(be, dst, bytes);
    std::lock_guard<std::mutex> g(be->stage_mu);
    const char *at;
    if (rc = stage_upload(be, src_host, bytes, &at); rc) return rc;
    VX_CHECK_HIP(hipMemcpyAsync(dst, at, bytes, hipMemcpyHostToDevice, be->stream));
    return VX_OK;
}

// What bounds a step's small uploads is the host: each copy of the runtime's is 6 us of it, 66 of them (the tables of 32 sequences
// that have all come to a new block) 400 us before the step's first kernel. One launch brings 64.
int vx_to_device_staged_many(vx_backend *be, int n, void *const *dst, const void *const *src_host, const size_t *bytes) {
    int rc = enter(be);
    if (rc) return rc;
    if (n == 0) return VX_OK;
    VX_REQUIRE(n > 0 && dst && src_host && bytes, "vx_to_device_staged: bad arguments");
    VX_REQUIRE(!be->capturing, "vx_to_device_staged during graph capture");
    int small = 0;
    for (int i = 0; i < n; i++) {
        VX_REQUIRE(!dst[i] || bytes[i] == 0 || src_host[i] != nullptr, "vx_to_device_staged: null source");
        small += dst[i] && bytes[i] > 0 && bytes[i] <= UP_MOST;
    }
    if (small <= 2) {
        for (int i = 0; i < n; i++)
            if (rc = vx_to_device_staged(be, dst[i], src_host[i], bytes[i]); rc) return rc;
        return VX_OK;
    }
    ScatterArgs a;
    int m = 0;
    size_t used = 0;  // of the staging memory, by the launch in the making
    std::unique_lock<std::mutex> g(be->stage_mu);
    auto launch = [&]() -> int {
        if (m == 0) return VX_OK;
        scatter_kernel<<<m, SEND_THREADS, 0, be->stream>>>(a);
        be->stage_used += used;
        m = 0, used = 0;
        VX_CHECK_LAUNCH();
        return VX_OK;
    };
    for (int i = 0; i < n; i++) {
        if (!dst[i] || bytes[i] == 0) continue;
        if (bytes[i] > UP_MOST || !device_memory(be, dst[i], bytes[i])) {
            if (rc = launch(); rc) return rc;
            g.unlock();
            if (rc = vx_to_device_staged(be, dst[i], src_host[i], bytes[i]); rc) return rc;
            g.lock();
            continue;
        }
        const size_t room = (bytes[i] + 63) / 64 * 64;
        if (m == SCATTER_MOST || be->stage_used + used + room > UP_BYTES)
            if (rc = launch(); rc) return rc;
        if (be->stage_used + room > UP_BYTES) {
            VX_CHECK_HIP(hipStreamSynchronize(be->stream));
            be->stage_used = 0;
        }
        if (m == 0) a.from = (const char *)be->host_stage + UP_AT + be->stage_used;
        items_written(be, dst[i], bytes[i]);
        memcpy((char *)be->host_stage + UP_AT + be->stage_used + used, src_host[i], bytes[i]);
        a.dst[m] = (char *)dst[i], a.at[m] = (uint32_t)used, a.bytes[m] = (uint32_t)bytes[i];
        m++, used += room;
    }
    return launch();
}

}  // extern "C"
