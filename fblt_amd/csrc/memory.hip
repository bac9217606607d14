/*
 * Device-memory shim of the HIP backend: the functions the reference's core
 * calls for device arenas and tensor transfers (reference contract:
 * csrc/core/cuda_shim.h:18-31; behaviour: csrc/ops/memory.cu:37-77).  Memset
 * and host-to-device copies are asynchronous on the library's current stream
 * (the null stream unless blt_hip_set_stream chose another); the
 * device-to-host copy blocks and is the implicit synchronisation point.
 */
#include "blt_hip.h"
#include "blt_fatal.h"
#include "hip_check.h"
#include "launch.h"

#include <algorithm>
#include <stdint.h>

extern "C" void *blt_hip_malloc(size_t bytes) {
    void *p = nullptr;
    HIP_CHECK(hipMalloc(&p, bytes));
    return p;
}

extern "C" void blt_hip_free(void *ptr) {
    if (!ptr) return;
    hipError_t e = hipFree(ptr);
    if (e != hipSuccess) BLT_WARN("HIP hipFree failed: %s", hipGetErrorString(e));
}

namespace {

/* Byte fill as a kernel: 16-byte stores over the aligned body, single bytes at the ragged ends. */
__global__ __launch_bounds__(256) void fill_bytes_kernel(unsigned char *dst, unsigned int pattern, size_t head,
                                                         size_t body16, size_t bytes) {
    const size_t t = (size_t)blockIdx.x * 256u + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * 256u;
    uint4 *body = reinterpret_cast<uint4 *>(dst + head);
    for (size_t i = t; i < body16; i += stride) body[i] = make_uint4(pattern, pattern, pattern, pattern);
    const size_t tail0 = head + 16u * body16;
    for (size_t i = t; i < head; i += stride) dst[i] = (unsigned char)pattern;
    for (size_t i = tail0 + t; i < bytes; i += stride) dst[i] = (unsigned char)pattern;
}

} // namespace

/* While a graph is being captured the fill is a kernel node: memset nodes recorded into a graph
 * have replayed wrongly on this platform, and blt_tensor_create (zero-filled tensors) reaches this
 * from inside captured calls. */
extern "C" void blt_hip_memset(void *dst, int value, size_t bytes) {
    if (bytes == 0) return;
    if (!blt_stream_capturing()) {
        HIP_CHECK(hipMemsetAsync(dst, value, bytes, blt_stream()));
        return;
    }
    const uintptr_t addr = reinterpret_cast<uintptr_t>(dst);
    const size_t head = std::min<size_t>(bytes, (16u - (addr & 15u)) & 15u);
    const size_t body16 = (bytes - head) / 16u;
    const unsigned int b = (unsigned int)(value & 0xFF), pattern = b | (b << 8) | (b << 16) | (b << 24);
    const unsigned blocks = (unsigned)std::min<size_t>(2048, std::max<size_t>(1, (body16 + 255) / 256));
    blt_launch("fill_bytes", fill_bytes_kernel, dim3(blocks), dim3(256), 0, blt_stream(), static_cast<unsigned char *>(dst),
               pattern, head, body16, bytes);
    HIP_CHECK_LAUNCH("blt_hip_memset");
}


namespace {

/* Ring of pinned buffers, one event each: a slot is reused only after the copy
 * that read it has finished. */
struct PinnedRing {
    static constexpr int SLOTS = 8;
    struct Slot {
        void *host = nullptr;
        size_t capacity = 0;
        hipEvent_t copied = nullptr;
        bool in_flight = false;
    } slot[SLOTS];
    int next = 0;
};

/* Small uploads travel in the argument block of a kernel that writes them out: the copy engine's way, pinned buffer and
 * event included, keeps the stream for about 15 us between two kernels, a launch for about 4 (and there is nothing
 * to wait for before the source may change).  Words that fit 16 bits travel as such: row ranges and lengths do. */
constexpr size_t ARG_WORDS = 992; /* 3968 of an argument block's 4096 bytes */
struct UploadArgs {
    uint32_t *dst;
    uint32_t count;
    uint32_t halves; /* two words of 16 bits in each */
    uint32_t words[ARG_WORDS];
};
static_assert(sizeof(UploadArgs) <= 4096, "kernel argument block");
__global__ __launch_bounds__(256) void upload_words_kernel(UploadArgs a) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= a.count) return;
    a.dst[i] = a.halves ? (a.words[i >> 1] >> (16u * (i & 1u))) & 0xFFFFu : a.words[i];
}

/* false: more than two launches' worth, the copy engine is level from there on */
bool upload_in_arguments(void *dst, const void *src, size_t bytes) {
    if ((bytes & 3u) != 0 || (reinterpret_cast<uintptr_t>(dst) & 3u) != 0 || (reinterpret_cast<uintptr_t>(src) & 3u) != 0 ||
        bytes > 4u * ARG_WORDS * 4u)
        return false;
    const uint32_t *from = static_cast<const uint32_t *>(src);
    const size_t count = bytes / 4u;
    uint32_t any = 0;
    for (size_t i = 0; i < count; i++) any |= from[i];
    const bool halves = any <= 0xFFFFu;
    const size_t per_launch = halves ? 2u * ARG_WORDS : ARG_WORDS;
    if (count > 2u * per_launch) return false;
    UploadArgs a;
    a.halves = halves ? 1u : 0u;
    for (size_t at = 0; at < count; at += per_launch) {
        a.dst = static_cast<uint32_t *>(dst) + at;
        a.count = (uint32_t)(count - at < per_launch ? count - at : per_launch);
        if (halves) {
            for (uint32_t i = 0; i < a.count; i += 2u)
                a.words[i / 2u] = from[at + i] | (i + 1u < a.count ? from[at + i + 1u] << 16 : 0u);
        } else {
            __builtin_memcpy(a.words, from + at, 4u * a.count);
        }
        blt_launch("upload_words", upload_words_kernel, dim3((a.count + 255u) / 256u), dim3(256), 0, blt_stream(), a);
    }
    HIP_CHECK_LAUNCH("upload_words");
    return true;
}

} // namespace

void blt_upload_staged(void *dst, const void *src, size_t bytes) {
    if (bytes == 0) return;
    BLT_REQUIRE(!blt_stream_capturing(), "host data cannot be staged to the device while a graph is captured");
    if (upload_in_arguments(dst, src, bytes)) return;
    /* a replay would copy what the ring's buffer holds by then, and an event recorded there cannot be waited for */
    BLT_REQUIRE(!blt_stream_captured_by_caller(),
                "more host data than launch arguments hold cannot be staged to the device while the stream is captured");
    static thread_local PinnedRing ring;
    PinnedRing::Slot &s = ring.slot[ring.next];
    ring.next = (ring.next + 1) % PinnedRing::SLOTS;
    if (!s.copied) HIP_CHECK(hipEventCreateWithFlags(&s.copied, hipEventDisableTiming));
    if (s.in_flight) {
        HIP_CHECK(hipEventSynchronize(s.copied));
        s.in_flight = false;
    }
    if (bytes > s.capacity) {
        if (s.host) HIP_CHECK(hipHostFree(s.host));
        s.capacity = bytes < 32768 ? 65536 : 2 * bytes; /* few re-allocations: pinning memory costs ~100 us */
        HIP_CHECK(hipHostMalloc(&s.host, s.capacity, hipHostMallocDefault));
    }
    __builtin_memcpy(s.host, src, bytes);
    HIP_CHECK(hipMemcpyAsync(dst, s.host, bytes, hipMemcpyHostToDevice, blt_stream()));
    HIP_CHECK(hipEventRecord(s.copied, blt_stream()));
    s.in_flight = true;
}

/* The reference's callers free or reuse the host buffer as soon as the upload call returns
 * (csrc/infer/kv_cache.c:237-238), so the source must be consumed before this returns: small
 * uploads go through the pinned ring (no wait), large ones wait for the copy. */
extern "C" void blt_hip_memcpy_h2d(void *dst, const void *src, size_t bytes) {
    if (bytes == 0) return;
    if (bytes <= (1u << 20) && !blt_stream_capturing()) {
        blt_upload_staged(dst, src, bytes);
        return;
    }
    HIP_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, blt_stream()));
    HIP_CHECK(hipStreamSynchronize(blt_stream()));
}

extern "C" void blt_hip_memcpy_d2h(void *dst, const void *src, size_t bytes) {
    if (bytes == 0) return;
    /* the copy waits for the library's current stream, whichever it is */
    HIP_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, blt_stream()));
    HIP_CHECK(hipStreamSynchronize(blt_stream()));
    blt_kv_check_device_errors();
}

extern "C" void blt_backend_pass_sync_hip(void) {
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e != hipSuccess) BLT_FATAL("blt_backend_pass_sync: %s", hipGetErrorString(e));
    blt_kv_check_device_errors();
}

extern "C" const char *blt_hip_build_info(void) { return "fblt_amd attention backend; kernels: gfx950"; }
