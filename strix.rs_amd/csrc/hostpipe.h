// Large host-pointer transfers: activations in from and results out to the caller's pageable memory.
//
// A copy between the device and pageable memory runs at 10 - 18 GB/s on this path: the runtime stages it through its own
// buffers on one thread, and a result array the caller has just allocated is faulted in page by page on the way (14 GB/s by
// itself).  The bus carries 57 GB/s each way.  HostPipe cuts a transfer into pieces that pass through a ring of pinned
// buffers on streams of their own (one per direction, default priority), a few worker threads move the pieces between the
// ring and the caller's memory, and the result's pages are populated by the same threads while the device is still busy.
// Outbound, a copy command per piece with an event behind it would cost 13 us of idle bus each (2 MB pieces: 41 GB/s, 8 MB:
// 52); a kernel of kOutWgs small workgroups writes pinned memory at 54 GB/s from 16 CUs on, and says in pinned memory which
// 16 KB parts have arrived, so that the last part is on its way to the caller microseconds after it has left the device.
// Bound: the bus (1024 x 9728 results of a 2560-long GEMM: 40 MB out = 0.74 of the call's 1.08 ms; 4.4 ms with pageable copies).
//
// Owned by one context, made by its first large call, given back with it: at most kMaxWorkers threads (asleep between
// calls, and within one when they have found no work for kSpinUs: the device computes) and kInSlots * kPiece + kOutRing bytes
// of pinned memory, whatever the call's size.  Making it costs that first call: 190 x 4096 results of 256-long rows 7.8 ms in a
// fresh process and 1.3 - 1.6 ms in a later context, where the second call takes 0.22 - 0.5; 700 rows 2.7 - 3.4 ms against 0.6.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstddef>
#include <mutex>
#include <thread>
#include <vector>

struct smx_ctx;

namespace smx {

class HostPipe {
public:
    static constexpr size_t kPiece = size_t(2) << 20;     // one inbound transfer
    static constexpr size_t kTask = size_t(256) << 10;    // one worker's copy
    static constexpr int kInSlots = 8;
    static constexpr size_t kPart = size_t(16) << 10;     // outbound: what one workgroup copies and reports
    static constexpr size_t kOutRing = size_t(48) << 20;
    static constexpr size_t kMaxSpan = size_t(12) << 20;  // outbound: one launch
    static constexpr int kMaxSpans = 64;
    static constexpr unsigned kOutWgs = 32;
    static constexpr int kMaxWorkers = 5;                 // more bring nothing: the bus is the bound
    static constexpr double kSpinUs = 250.0;              // a call's own gaps are shorter (50: 1024 x 9728 results 2 % slower; 250: as without sleep)
    static constexpr int kQueue = 4096;

    ~HostPipe();
    int open(smx_ctx* c);      // threads, streams, events, ring: once
    // A call's transfers lie between begin and end.  begin: the transfers follow what is queued on the context's stream.
    int begin(smx_ctx* c);
    // Populate the pages of a result array in the background (its contents stay as they are).
    void populate(void* host, size_t bytes);
    // Copy in, in order, on the inbound stream; the context's stream waits for everything sent so far with in_done.
    int in(smx_ctx* c, void* dev, const void* host, size_t bytes);
    int in_done(smx_ctx* c);
    // Copy out what the context's stream has produced so far.
    int out(smx_ctx* c, void* host, const void* dev, size_t bytes);
    int end(smx_ctx* c, int rc);   // every transfer has landed (also after an error: nothing touches the caller's memory any more)

private:
    struct Task {
        char* dst;
        const char* src;   // null: populate dst
        size_t n;
        std::atomic<int>* left;
    };
    struct Span {   // one outbound launch: n bytes at ring offset `off`, on their way to host
        size_t off, n, handed;   // handed: bytes given to the workers
        char* host;
        unsigned seq;            // what its parts report
        std::atomic<int> left;   // copies still to do
    };
    struct Queue {   // single producer (the calling thread), many consumers
        std::vector<Task> task;
        std::atomic<size_t> head{0}, tail{0}, done{0};
    };
    void worker();
    bool waiting(const Queue& q) const { return q.head.load() < q.tail.load(); }
    bool run_one(Queue& q);
    void push(Queue& q, char* dst, const char* src, size_t n, std::atomic<int>* left);
    void push_copies(char* dst, const char* src, size_t n, std::atomic<int>* left);
    int progress(smx_ctx* c);
    int wait_progress(smx_ctx* c);
    bool ring_room(size_t n, size_t* off);

    int device = 0;
    hipStream_t s_in = nullptr, s_out = nullptr;
    hipEvent_t ev_in[kInSlots] = {}, ev_mark = nullptr;
    char *ring_in = nullptr, *ring_out = nullptr;
    unsigned* flags = nullptr;       // pinned: one word per part of the outbound ring
    bool in_used[kInSlots] = {};
    unsigned next_in = 0;
    Span spans[kMaxSpans];
    size_t span_first = 0, span_handing = 0, span_end = 0;   // spans[i % kMaxSpans]: freed < first <= handing <= end
    size_t ring_head = 0;            // where the next span goes
    unsigned seq = 0;
    std::chrono::steady_clock::time_point last_progress;

    Queue copies, pages;   // pages (populate) are taken when no copy waits, and never by the calling thread before the end
    std::atomic<int> sleepers{0};
    unsigned calls = 0;              // under mu, as quit: what a sleeping worker also wakes for
    bool quit = false;
    std::mutex mu;
    std::condition_variable cv;
    std::vector<std::thread> threads;
};

}  // namespace smx
