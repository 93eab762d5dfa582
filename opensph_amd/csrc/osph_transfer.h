// Device results to the host (osph_transfer.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace osph {

// Copies device memory written by earlier work on `stream` into host memory, and returns when it is there.
// Safe from several threads and for several streams and devices (the calling thread's current one).
hipError_t copy_to_host(hipStream_t stream, void* host, const void* dev, size_t bytes);
// Every context that copies is attached while it lives; the pinned buffers go with the last one.
void transfer_attach();
void transfer_detach();

// A few 64-bit words of device memory to the host in the middle of a chain of launches.  host[0 .. words) are pinned and
// coherent, host[words] counts the posts; a kernel at its place in the stream writes the words, then the count, and the
// waiting thread watches the count.  A copy command and the wait for the stream leave the device idle for 10 to 20 us
// each time: steps of 2k / 40k particles 110 / 155 -> 94 / 148 us (two waits each), a Barnes-Hut step of 20k particles
// 447 -> 370 us (four waits -> three).  Words written by the last reducing kernel itself instead of k_post: no gain, its
// blocks' fences to the host cost what the launch does.
struct Mailbox {
    unsigned long long* host = nullptr;
    size_t words = 0;
    unsigned long long posts = 0;
};
hipError_t mailbox_create(Mailbox& box, size_t words);
void mailbox_destroy(Mailbox& box);  // the stream must be idle
// For a kernel that writes host words itself: their place, and the count to store behind them.
struct MailboxPost {
    unsigned long long* host;
    unsigned long long* posts;
    unsigned long long value;
};
MailboxPost mailbox_next(Mailbox& box);
// Queues dev[0 .. count) -> host[first ..).
void mailbox_post(hipStream_t stream, Mailbox& box, size_t first, const unsigned long long* dev, size_t count);
// Waits for everything posted so far (and so for all earlier work of the stream).
hipError_t mailbox_wait(hipStream_t stream, Mailbox& box);

}  // namespace osph
