// Device results into the caller's host memory, pageable as a rule.
//
// hipMemcpyAsync into pageable memory goes through the runtime's staging buffer, 1 MB at a time: each megabyte is
// copied by the device (20 us), then by one host thread, about 12 GB/s in all.  Here the pieces go through pinned
// buffers of this library with the device copy of the next piece running while the last one is copied out, on up to
// COPY_THREADS host threads, each with its own range and its own two half buffers.  Measured
// (runtime's copy -> this, 500k x 32 B, 4M x 32 B, 2k x 32 B): 900 -> 565 us, 7235 -> 3330 us, 52 -> 35 us, so 28 and
// 38 GB/s.  Pieces of 512 KB, 1 MB, 4 MB: 650, 617, 534 us for the first size; the pinned memory (4 MB a buffer, once
// per process, 0.7 ms each) sets the limit upwards.  6 and 8 threads are no faster than 4.
#include "osph_transfer.h"

#include <algorithm>
#include <chrono>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace osph {
namespace {

constexpr size_t PIECE = size_t(2) << 20;  // bytes of half a pinned buffer
constexpr int COPY_THREADS = 4;
constexpr size_t MAX_BUFFERS = 8;          // pinned buffers of the process (32 MB)
constexpr size_t THREAD_BYTES = size_t(2) << 20;  // a further thread for every so many bytes

struct PinnedBuffer {
    unsigned char* mem = nullptr;  // two pieces
    hipEvent_t done[2] = { nullptr, nullptr };
    int device = -1;
};

// The pinned buffers of the process: at most MAX_BUFFERS, shared by all contexts, each in the hands of one thread at
// a time, freed when the last context goes.
struct PinnedPool {
    std::mutex lock;
    std::vector<PinnedBuffer> idle;
    size_t made = 0, users = 0;
};

PinnedPool& pool() {
    static PinnedPool p;
    return p;
}

void destroy_events(PinnedBuffer& b) {
    for (hipEvent_t& e : b.done) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
}

void destroy_buffer(PinnedBuffer& b) {
    destroy_events(b);
    if (b.mem) (void)hipHostFree(b.mem);
    b = PinnedBuffer{};
}

// A buffer whose events belong to `device`: an idle one of that device, a new one, or at the limit an idle one of another
// device (the memory serves all, the events are made anew).  False when all are in use or something cannot be
// allocated (the caller then copies without one).
bool take_buffer(int device, PinnedBuffer& out) {
    PinnedPool& p = pool();
    PinnedBuffer b;
    {
        std::lock_guard<std::mutex> g(p.lock);
        size_t k = 0;
        while (k < p.idle.size() && p.idle[k].device != device) ++k;
        if (k == p.idle.size() && p.made < MAX_BUFFERS) {
            ++p.made;
        } else if (!p.idle.empty()) {
            k = std::min(k, p.idle.size() - 1);
            b = p.idle[k];
            p.idle.erase(p.idle.begin() + long(k));
        } else {
            return false;
        }
    }
    const hipError_t before = hipPeekAtLastError();
    if (b.device != device) destroy_events(b);
    b.device = device;
    bool made = b.mem || hipHostMalloc(reinterpret_cast<void**>(&b.mem), 2 * PIECE, hipHostMallocPortable) == hipSuccess;
    for (hipEvent_t& e : b.done) made = made && (e || hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess);
    if (made) {
        out = b;
        return true;
    }
    if (before == hipSuccess) (void)hipGetLastError();  // an earlier error stays
    destroy_buffer(b);
    std::lock_guard<std::mutex> g(p.lock);
    --p.made;
    return false;
}

void give_buffer(PinnedBuffer& b) {
    PinnedPool& p = pool();
    std::unique_lock<std::mutex> g(p.lock);
    if (p.users > 0) {
        p.idle.push_back(b);  // capacity reserved in transfer_attach
        return;
    }
    --p.made;
    g.unlock();
    destroy_buffer(b);
}

// bytes [0, n) of dev into host through b, piece by piece: the device fills one half while the other is copied out.
hipError_t copy_range(hipStream_t stream, PinnedBuffer& b, unsigned char* host, const unsigned char* dev, size_t n) {
    const size_t pieces = (n + PIECE - 1) / PIECE;
    hipError_t err = hipSuccess;
    size_t queued = 0;
    for (size_t k = 0; k < pieces && err == hipSuccess; ++k) {
        for (; queued < pieces && queued < k + 2 && err == hipSuccess; ++queued) {
            const size_t at = queued * PIECE;
            err = hipMemcpyAsync(b.mem + (queued & 1) * PIECE, dev + at, std::min(PIECE, n - at), hipMemcpyDeviceToHost,
                                 stream);
            if (err == hipSuccess) err = hipEventRecord(b.done[queued & 1], stream);
        }
        if (err == hipSuccess) err = hipEventSynchronize(b.done[k & 1]);
        if (err == hipSuccess) std::memcpy(host + k * PIECE, b.mem + (k & 1) * PIECE, std::min(PIECE, n - k * PIECE));
    }
    if (err != hipSuccess) (void)hipStreamSynchronize(stream);  // nothing may still write into the buffer
    return err;
}

// Whether the runtime knows the memory (allocated or registered through it), so that the device can copy to it itself.
bool known_memory(const void* p) {
    const hipError_t before = hipPeekAtLastError();
    hipPointerAttribute_t at{};
    if (hipPointerGetAttributes(&at, p) == hipSuccess) return at.type != hipMemoryTypeUnregistered;
    if (before == hipSuccess) (void)hipGetLastError();  // an earlier error stays
    return false;
}

__global__ void __launch_bounds__(256) k_post(const unsigned long long* __restrict__ src, size_t count,
                                              unsigned long long* __restrict__ host, unsigned long long* __restrict__ posts,
                                              unsigned long long value) {
    for (size_t k = threadIdx.x; k < count; k += blockDim.x) {
        __hip_atomic_store(host + k, src[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(posts, value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Watching the count costs a core its time: past this the thread sleeps in the runtime's wait, which is what a device
// error ends too.
constexpr std::chrono::milliseconds WATCH{ 20 };

}  // namespace

hipError_t mailbox_create(Mailbox& box, size_t words) {
    box = Mailbox{};
    const hipError_t e = hipHostMalloc(reinterpret_cast<void**>(&box.host), (words + 1) * sizeof(unsigned long long),
                                       hipHostMallocCoherent | hipHostMallocPortable | hipHostMallocMapped);
    if (e != hipSuccess) {
        box.host = nullptr;
        return e;
    }
    box.words = words;
    std::fill(box.host, box.host + words + 1, 0ull);
    return hipSuccess;
}

void mailbox_destroy(Mailbox& box) {
    if (box.host) (void)hipHostFree(box.host);
    box = Mailbox{};
}

MailboxPost mailbox_next(Mailbox& box) { return { box.host, box.host + box.words, ++box.posts }; }

void mailbox_post(hipStream_t stream, Mailbox& box, size_t first, const unsigned long long* dev, size_t count) {
    k_post<<<1, count > 64 ? 256 : 64, 0, stream>>>(dev, count, box.host + first, box.host + box.words, ++box.posts);
}

hipError_t mailbox_wait(hipStream_t stream, Mailbox& box) {
    const auto end = std::chrono::steady_clock::now() + WATCH;
    while (__atomic_load_n(box.host + box.words, __ATOMIC_ACQUIRE) != box.posts) {
        for (int k = 0; k < 16; ++k) __builtin_ia32_pause();
        if (std::chrono::steady_clock::now() < end) continue;
        if (const hipError_t e = hipStreamSynchronize(stream)) return e;
        if (__atomic_load_n(box.host + box.words, __ATOMIC_ACQUIRE) == box.posts) break;
        return hipErrorLaunchFailure;  // the stream is idle and a post is missing
    }
    return hipSuccess;
}

void transfer_attach() {
    PinnedPool& p = pool();
    std::lock_guard<std::mutex> g(p.lock);
    ++p.users;
    p.idle.reserve(MAX_BUFFERS);
}

void transfer_detach() {
    PinnedPool& p = pool();
    std::lock_guard<std::mutex> g(p.lock);
    if (--p.users > 0) return;
    for (PinnedBuffer& b : p.idle) destroy_buffer(b);
    p.made -= p.idle.size();
    p.idle.clear();
}

hipError_t copy_to_host(hipStream_t stream, void* host, const void* dev, size_t bytes) {
    if (!bytes) return hipSuccess;
    int device = 0;
    if (hipError_t e = hipGetDevice(&device)) return e;
    auto direct = [&]() -> hipError_t {
        if (hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, stream)) return e;
        return hipStreamSynchronize(stream);
    };
    // into the caller's pinned memory the device copies at the link's rate: 70k x 32 B 64 us, 1M x 32 B 617 us, where the
    // pieces below take 148 and 927 us
    if (known_memory(host)) return direct();
    const size_t hw = std::max<size_t>(std::thread::hardware_concurrency(), 1);
    const size_t want = std::min({ size_t(COPY_THREADS), hw, bytes / THREAD_BYTES + 1 });
    PinnedBuffer buf[COPY_THREADS];
    size_t parts = 0;
    while (parts < want && take_buffer(device, buf[parts])) ++parts;
    if (parts == 0) return direct();
    // whole pieces per part
    const size_t share = ((bytes + parts - 1) / parts + PIECE - 1) / PIECE * PIECE;
    hipError_t errs[COPY_THREADS];
    auto part = [&](size_t k) {
        const size_t at = std::min(k * share, bytes), n = std::min(share, bytes - at);
        errs[k] = n ? copy_range(stream, buf[k], static_cast<unsigned char*>(host) + at,
                                 static_cast<const unsigned char*>(dev) + at, n)
                    : hipSuccess;
    };
    std::thread others[COPY_THREADS];
    size_t started = 1;
    for (; started < parts; ++started) {
        const size_t k = started;
        try {
            others[k] = std::thread([&, k] {
                errs[k] = hipSetDevice(device);
                if (errs[k] == hipSuccess) part(k);
            });
        } catch (const std::exception&) {
            break;  // no further thread, or no memory for one: this one does the rest
        }
    }
    part(0);
    for (size_t k = started; k < parts; ++k) part(k);
    for (size_t k = 1; k < started; ++k) others[k].join();
    hipError_t err = hipSuccess;
    for (size_t k = 0; k < parts; ++k) {
        if (err == hipSuccess) err = errs[k];
        give_buffer(buf[k]);
    }
    return err;
}

}  // namespace osph
