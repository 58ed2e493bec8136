// Copies between host and device memory. C ABI: include/vexel_hip.h.
//
// A step of a model gives its caller megabytes of logits in ordinary (pageable) memory, often memory that has just been
// allocated and is not there yet. The runtime's own copy of that kind moves a piece at a time through a buffer of its own and
// copies (and takes the page faults of) each on the calling thread: 32 MiB take 3.4 ms where the bus needs 0.6 ms.
// Here the pieces go through a ring of pinned memory one behind the other, and a few threads of the backend copy
// those that have arrived while later ones are on their way. Small uploads go through pinned memory without waiting.
#include "common.h"
#include "transfer_ring.h"

namespace vx {

void mover_destroy(Mover *m) { delete m; }

// The backend's pinned megabyte: a word of vx_argmax's, staged uploads, small downloads.
constexpr size_t UP_AT = 64 << 10, UP_BYTES = 448 << 10, DOWN_AT = 512 << 10, DOWN_BYTES = 512 << 10, UP_MOST = 64 << 10;

static int download(vx_backend *be, int n, void *const *dst, const void *const *src, const size_t *bytes) {
    size_t total = 0;
    for (int i = 0; i < n; i++)
        if (src[i]) total += (bytes[i] + 63) / 64 * 64;
    if (total == 0) return VX_OK;
    for (int i = 0; i < n; i++) VX_REQUIRE(!src[i] || bytes[i] == 0 || dst[i] != nullptr, "vx_to_host: null destination");
    if (total <= DOWN_BYTES) {
        std::lock_guard<std::mutex> g(be->stage_mu);
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
    Mover *mover = nullptr;
    if (!pinned) {
        std::lock_guard<std::mutex> g(be->stage_mu);
        if (!be->mover) {
            be->mover = new Mover();
            if (!be->mover->start(std::min<int>(Mover::MAX_WORKERS, std::max(1u, std::thread::hardware_concurrency()) - 1))) {
                delete be->mover;
                be->mover = nullptr;
                (void)hipGetLastError();
            }
        }
        mover = be->mover;
    }
    if (!mover) {
        for (int i = 0; i < n; i++)
            if (src[i] && bytes[i] > 0) VX_CHECK_HIP(hipMemcpyAsync(dst[i], src[i], bytes[i], hipMemcpyDeviceToHost, be->stream));
        VX_CHECK_HIP(hipStreamSynchronize(be->stream));
        return VX_OK;
    }
    // pieces of an eighth, so that the threads have something to share, of 256 KiB to a slot
    const size_t most = std::min(Mover::SLOT, std::max((size_t)256 << 10, total / 8 / 4096 * 4096));
    std::vector<Mover::Piece> pieces;
    for (int i = 0; i < n; i++) {
        if (!src[i]) continue;
        for (size_t at = 0; at < bytes[i]; at += most)
            pieces.push_back({(char *)dst[i] + at, (const char *)src[i] + at, std::min(most, bytes[i] - at)});
    }
    std::lock_guard<std::mutex> g(mover->call);
    Mover::Job job(std::move(pieces));
    VX_CHECK_HIP(mover->move(be->stream, job));
    return VX_OK;
}

}  // namespace vx

using namespace vx;

extern "C" {

int vx_to_host_many(vx_backend *be, int n, void *const *dst_host, const void *const *src, const size_t *bytes) {
    int rc = enter(be);
    if (rc) return rc;
    if (n == 0) return VX_OK;
    VX_REQUIRE(n > 0 && dst_host && src && bytes, "vx_to_host: bad arguments");
    VX_REQUIRE(!be->capturing, "vx_to_host during graph capture");
    try {
        rc = download(be, n, dst_host, src, bytes);
    } catch (...) {
        set_error("vx_to_host: out of host memory");
        return VX_ERR_OOM;
    }
    return rc;
}

int vx_to_host(vx_backend *be, void *dst_host, const void *src, size_t bytes) {
    int rc = enter(be);
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
    const size_t room = (bytes + 63) / 64 * 64;
    std::lock_guard<std::mutex> g(be->stage_mu);
    if (be->stage_used + room > UP_BYTES) {
        VX_CHECK_HIP(hipStreamSynchronize(be->stream));
        be->stage_used = 0;
    }
    char *at = (char *)be->host_stage + UP_AT + be->stage_used;
    be->stage_used += room;
    memcpy(at, src_host, bytes);
    VX_CHECK_HIP(hipMemcpyAsync(dst, at, bytes, hipMemcpyHostToDevice, be->stream));
    return VX_OK;
}

}  // extern "C"
