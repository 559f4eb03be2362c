// Large host-pointer transfers (see hostpipe.h).
#include "hostpipe.h"

#include <emmintrin.h>
#include <sched.h>
#include <sys/mman.h>

#include <algorithm>
#include <cstring>
#include <system_error>

#include "smx_internal.h"

#ifndef MADV_POPULATE_WRITE
#define MADV_POPULATE_WRITE 23
#endif

namespace smx {

// Neither side is read again soon: streaming stores keep the destination from being fetched first and the caches for the
// pages the kernel has just cleared (fresh results 1.14 -> 1.10 ms, kept ones 0.97 -> 0.96 at 40 MB).
static void copy_streaming(char* dst, const char* src, size_t n) {
    if ((((uintptr_t)dst | (uintptr_t)src) & 15) != 0) {
        std::memcpy(dst, src, n);
        return;
    }
    const __m128i* s = (const __m128i*)src;
    __m128i* d = (__m128i*)dst;
    size_t i = 0;
    for (; i + 4 <= n / 16; i += 4) {
        const __m128i a = _mm_load_si128(s + i), b = _mm_load_si128(s + i + 1), c = _mm_load_si128(s + i + 2), e = _mm_load_si128(s + i + 3);
        _mm_stream_si128(d + i, a);
        _mm_stream_si128(d + i + 1, b);
        _mm_stream_si128(d + i + 2, c);
        _mm_stream_si128(d + i + 3, e);
    }
    std::memcpy(dst + i * 16, src + i * 16, n - i * 16);
    _mm_sfence();
}

bool HostPipe::run_one(Queue& q) {
    size_t h = q.head.load(std::memory_order_relaxed);
    while (h < q.tail.load(std::memory_order_acquire)) {
        if (!q.head.compare_exchange_weak(h, h + 1, std::memory_order_acq_rel)) continue;
        const Task t = q.task[h % kQueue];   // not overwritten before `done` has counted it
        if (t.src) copy_streaming(t.dst, t.src, t.n);
        else (void)madvise(t.dst, t.n, MADV_POPULATE_WRITE);   // a hint: the copy faults the pages in where it is not known
        if (t.left) t.left->fetch_sub(1, std::memory_order_release);
        q.done.fetch_add(1, std::memory_order_release);
        return true;
    }
    return false;
}

void HostPipe::worker() {
    unsigned seen = 0;
    auto idle = std::chrono::steady_clock::now();
    for (;;) {
        if (run_one(copies) || run_one(pages)) {
            idle = std::chrono::steady_clock::now();
            continue;
        }
        for (int i = 0; i < 32; i++) __builtin_ia32_pause();   // while transfers run the next task is microseconds away
        if (std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - idle).count() < kSpinUs) continue;
        std::unique_lock<std::mutex> l(mu);
        sleepers.fetch_add(1);   // in front of the look at the queues: a push either is seen there or sees the sleeper
        cv.wait(l, [&] { return quit || calls != seen || waiting(copies) || waiting(pages); });
        sleepers.fetch_sub(1);
        if (quit) return;
        seen = calls;
        idle = std::chrono::steady_clock::now();
    }
}

void HostPipe::push(Queue& q, char* dst, const char* src, size_t n, std::atomic<int>* left) {
    const size_t t = q.tail.load(std::memory_order_relaxed);
    while (t - q.done.load(std::memory_order_acquire) >= kQueue) run_one(q);
    q.task[t % kQueue] = Task{dst, src, n, left};
    q.tail.store(t + 1);
    if (sleepers.load() > 0) {
        { std::lock_guard<std::mutex> l(mu); }   // (not between a sleeper's look at the queues and its sleep)
        cv.notify_one();
    }
}

void HostPipe::push_copies(char* dst, const char* src, size_t n, std::atomic<int>* left) {
    left->store((int)((n + kTask - 1) / kTask), std::memory_order_relaxed);
    for (size_t o = 0; o < n; o += kTask) push(copies, dst + o, src + o, std::min(kTask, n - o), left);
}

int HostPipe::open(smx_ctx* c) {
    device = c->device;
    SMX_HIP(c, hipStreamCreateWithFlags(&s_in, hipStreamNonBlocking));
    SMX_HIP(c, hipStreamCreateWithFlags(&s_out, hipStreamNonBlocking));
    for (int i = 0; i < kInSlots; i++) SMX_HIP(c, hipEventCreateWithFlags(&ev_in[i], hipEventDisableTiming));
    SMX_HIP(c, hipEventCreateWithFlags(&ev_mark, hipEventDisableTiming));
    SMX_HIP(c, hipHostMalloc((void**)&ring_in, kInSlots * kPiece, kHostMemory));
    SMX_HIP(c, hipHostMalloc((void**)&ring_out, kOutRing, kHostMemory));
    SMX_HIP(c, hipHostMalloc((void**)&flags, kOutRing / kPart * 4, kHostMemory));
    std::memset(flags, 0, kOutRing / kPart * 4);   // sequence numbers start at 1
    copies.task.resize(kQueue);
    pages.task.resize(kQueue);
    // one thread per core this process may run on, up to kMaxWorkers besides the caller's
    cpu_set_t set;
    int cores = 1;
    if (sched_getaffinity(0, sizeof set, &set) == 0) cores = CPU_COUNT(&set);
    try {
        for (int i = 0; i < std::min(kMaxWorkers, cores - 1); i++) threads.emplace_back([this] { worker(); });
    } catch (const std::system_error&) {
        // no further thread to be had: with those there are (the calling thread takes part in any case)
    }
    return SMX_OK;
}

HostPipe::~HostPipe() {
    {
        std::lock_guard<std::mutex> l(mu);
        quit = true;
    }
    cv.notify_all();
    for (auto& t : threads) t.join();
    for (hipEvent_t e : ev_in)
        if (e) (void)hipEventDestroy(e);
    if (ev_mark) (void)hipEventDestroy(ev_mark);
    if (s_in) (void)hipStreamSynchronize(s_in);
    if (s_out) (void)hipStreamSynchronize(s_out);
    if (s_in) (void)hipStreamDestroy(s_in);
    if (s_out) (void)hipStreamDestroy(s_out);
    if (ring_in) (void)hipHostFree(ring_in);
    if (ring_out) (void)hipHostFree(ring_out);
    if (flags) (void)hipHostFree(flags);
}

int HostPipe::begin(smx_ctx* c) {
    span_first = span_handing = span_end = 0;
    ring_head = 0;
    last_progress = std::chrono::steady_clock::now();
    for (bool& u : in_used) u = false;
    {
        std::lock_guard<std::mutex> l(mu);
        calls++;
    }
    cv.notify_all();   // the first pieces are being queued by the time the workers are up
    SMX_HIP(c, hipEventRecord(ev_mark, c->stream));
    SMX_HIP(c, hipStreamWaitEvent(s_in, ev_mark, 0));
    return SMX_OK;
}

void HostPipe::populate(void* host, size_t bytes) {
    const uintptr_t page = 4096, huge = uintptr_t(2) << 20;
    const uintptr_t a = ((uintptr_t)host + page - 1) & ~(page - 1), b = ((uintptr_t)host + bytes) & ~(page - 1);
    for (uintptr_t p = a; p < b;) {   // pieces end at 2 MB boundaries: no two threads in one huge page
        const uintptr_t e = std::min(b, (p + huge) & ~(huge - 1));
        push(pages, (char*)p, nullptr, e - p, nullptr);
        p = e;
    }
}

int HostPipe::in(smx_ctx* c, void* dev, const void* host, size_t bytes) {
    // the pieces' copies are queued ahead of the transfers: slot i + 1 fills while slot i is being sent
    std::atomic<int> left[kInSlots];
    for (auto& l : left) l.store(0);
    const size_t n = (bytes + kPiece - 1) / kPiece;
    int rc = SMX_OK;
    size_t filled = 0;
    for (size_t i = 0; i < n && rc == SMX_OK; i++) {
        while (filled < n && filled < i + kInSlots) {
            const int s = (int)((next_in + filled) % kInSlots);
            if (in_used[s]) {   // its last transfer has left the ring
                if (filled > i && hipEventQuery(ev_in[s]) != hipSuccess) {
                    (void)hipGetLastError();
                    break;
                }
                hipError_t e = hipEventSynchronize(ev_in[s]);
                if (e != hipSuccess) { rc = hip_fail(c, e, "hipEventSynchronize"); break; }
                in_used[s] = false;
            }
            push_copies(ring_in + s * kPiece, (const char*)host + filled * kPiece, std::min(kPiece, bytes - filled * kPiece), &left[s]);
            filled++;
        }
        if (rc != SMX_OK) break;
        const int s = (int)((next_in + i) % kInSlots);
        while (left[s].load(std::memory_order_acquire) > 0)
            if (!run_one(copies) && (rc = progress(c)) != SMX_OK) break;
        if (rc != SMX_OK) break;
        hipError_t e = hipMemcpyAsync((char*)dev + i * kPiece, ring_in + s * kPiece, std::min(kPiece, bytes - i * kPiece), hipMemcpyHostToDevice, s_in);
        if (e == hipSuccess) e = hipEventRecord(ev_in[s], s_in);
        if (e != hipSuccess) rc = hip_fail(c, e, "hipMemcpyAsync(in)");
        in_used[s] = true;
    }
    for (auto& l : left)   // the counters live here
        while (l.load(std::memory_order_acquire) > 0) run_one(copies);
    next_in = (unsigned)((next_in + n) % kInSlots);
    return rc;
}

int HostPipe::in_done(smx_ctx* c) {
    SMX_HIP(c, hipEventRecord(ev_mark, s_in));
    SMX_HIP(c, hipStreamWaitEvent(c->stream, ev_mark, 0));
    return SMX_OK;
}

// Part p (kPart bytes, the last one shorter) of a span goes from src to dst by workgroup p % kOutWgs, which then reports it.
// A part's loads are all requested before its stores.  The stores are write-through at system scope and waited for before
// the barrier in front of the report, so a host that sees the report sees the bytes.
__global__ __launch_bounds__(256) void span_out_kernel(const char* __restrict__ src, char* __restrict__ dst, size_t n, unsigned* flags, unsigned seq) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    constexpr int PER = HostPipe::kPart / (256 * 16);   // 16-byte pieces per thread
    const size_t parts = (n + HostPipe::kPart - 1) / HostPipe::kPart;
    for (size_t p = blockIdx.x; p < parts; p += gridDim.x) {
        const size_t o = p * HostPipe::kPart, len = min(HostPipe::kPart, n - o);
        f4 v[PER];
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const size_t e = ((size_t)j * 256 + threadIdx.x) * 16;
            if (e + 16 <= len) v[j] = *(const f4*)(src + o + e);
        }
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const size_t e = ((size_t)j * 256 + threadIdx.x) * 16;
            if (e + 16 <= len) asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1" : : "v"(dst + o + e), "v"(v[j]) : "memory");
        }
        const size_t tail = len & ~size_t(15);
        if (threadIdx.x < (len - tail) / 4)
            __hip_atomic_store((unsigned*)(dst + o + tail) + threadIdx.x, ((const unsigned*)(src + o + tail))[threadIdx.x], __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_SYSTEM);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0) __hip_atomic_store(flags + p, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// hand arrived parts to the workers, in order; free spans whose copies are done
int HostPipe::progress(smx_ctx* c) {
    while (span_handing < span_end) {
        Span& sp = spans[span_handing % kMaxSpans];
        while (sp.handed < sp.n) {
            const size_t n = std::min(kTask, sp.n - sp.handed);
            const volatile unsigned* f = flags + (sp.off + sp.handed) / kPart;
            for (size_t i = 0; i < (n + kPart - 1) / kPart; i++)
                if (f[i] != sp.seq) goto waiting;
            std::atomic_thread_fence(std::memory_order_acquire);
            push(copies, sp.host + sp.handed, ring_out + sp.off + sp.handed, n, &sp.left);
            sp.handed += n;
        }
        span_handing++;
    }
waiting:
    while (span_first < span_handing && spans[span_first % kMaxSpans].left.load(std::memory_order_acquire) == 0) span_first++;
    (void)c;
    return SMX_OK;
}

// n bytes in one piece behind the newest span, in front of the oldest one
bool HostPipe::ring_room(size_t n, size_t* off) {
    if (span_end - span_first >= kMaxSpans) return false;
    if (span_first == span_end) ring_head = 0;
    size_t h = ring_head;
    if (span_first < span_end) {
        const size_t t = spans[span_first % kMaxSpans].off;
        if (h > t) {                      // used: [t, h)
            if (h + n > kOutRing) {
                if (n >= t) return false; // keep head and tail apart
                h = 0;
            }
        } else if (h + n >= t) {          // used: [t, end) and [0, h)
            return false;
        }
    }
    *off = h;
    return true;
}

int HostPipe::out(smx_ctx* c, void* host, const void* dev, size_t bytes) {
    SMX_HIP(c, hipEventRecord(ev_mark, c->stream));
    SMX_HIP(c, hipStreamWaitEvent(s_out, ev_mark, 0));
    for (size_t o = 0; o < bytes;) {
        const size_t n = std::min(kMaxSpan, bytes - o);
        const size_t room = (n + kPart - 1) & ~(kPart - 1);
        size_t off = 0;
        while (!ring_room(room, &off)) {
            int rc = wait_progress(c);
            if (rc != SMX_OK) return rc;
        }
        Span& sp = spans[span_end % kMaxSpans];
        sp.off = off;
        sp.n = n;
        sp.handed = 0;
        sp.host = (char*)host + o;
        sp.seq = ++seq;
        sp.left.store((int)((n + kTask - 1) / kTask), std::memory_order_relaxed);
        const unsigned parts = (unsigned)((n + kPart - 1) / kPart);
        hipLaunchKernelGGL(span_out_kernel, dim3(std::min(parts, kOutWgs)), dim3(256), 0, s_out, (const char*)dev + o, ring_out + off, n,
                           flags + off / kPart, sp.seq);
        SMX_HIP(c, hipGetLastError());
        span_end++;
        ring_head = off + room;
        o += n;
        int rc = progress(c);
        if (rc != SMX_OK) return rc;
    }
    return SMX_OK;
}

// One step of waiting for outbound spans.  Without any progress for kStallS the streams are asked what happened.
int HostPipe::wait_progress(smx_ctx* c) {
    constexpr double kStallS = 5.0;
    const size_t before = span_first * 4096 + spans[span_handing % kMaxSpans].handed / kTask;
    int rc = progress(c);
    if (rc != SMX_OK || run_one(copies)) return rc;
    const auto now = std::chrono::steady_clock::now();
    if (span_first * 4096 + spans[span_handing % kMaxSpans].handed / kTask != before || span_first == span_end) {
        last_progress = now;
    } else if (std::chrono::duration<double>(now - last_progress).count() > kStallS) {
        SMX_HIP(c, hipStreamSynchronize(c->stream));
        SMX_HIP(c, hipStreamSynchronize(s_out));
        last_progress = now;
        if (span_handing < span_end && (rc = progress(c)) == SMX_OK && span_handing < span_end)
            return fail(c, SMX_ERR_HIP, "host transfer: the device finished without reporting its results");
    }
    return SMX_OK;
}

int HostPipe::end(smx_ctx* c, int rc) {
    last_progress = std::chrono::steady_clock::now();
    while (rc == SMX_OK && span_handing < span_end) rc = wait_progress(c);
    for (Queue* q : {&copies, &pages})
        while (q->done.load(std::memory_order_acquire) < q->tail.load(std::memory_order_relaxed)) run_one(*q);
    if (rc != SMX_OK) {   // whatever is still queued ends before the call returns
        (void)hipStreamSynchronize(s_in);
        (void)hipStreamSynchronize(c->stream);
        (void)hipStreamSynchronize(s_out);
    }
    return rc;
}

__global__ __launch_bounds__(256) void span_in_kernel(const unsigned* __restrict__ src, unsigned* __restrict__ dst, size_t n) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n / 4; i += (size_t)gridDim.x * 256) ((uint4*)dst)[i] = ((const uint4*)src)[i];
    if (blockIdx.x == 0 && threadIdx.x < (n & 3)) dst[(n & ~size_t(3)) + threadIdx.x] = src[(n & ~size_t(3)) + threadIdx.x];
}

int staged_to_device(smx_ctx* c, void* dev, const void* staged, size_t bytes) {
    hipLaunchKernelGGL(span_in_kernel, dim3((unsigned)std::min<size_t>(64, (bytes + 4095) / 4096)), dim3(256), 0, c->stream,
                       (const unsigned*)staged, (unsigned*)dev, bytes / 4);
    SMX_HIP(c, hipGetLastError());
    return SMX_OK;
}

int host_send(smx_ctx* c, void* dev, const void* host, size_t bytes, bool read_once, void* result, size_t result_bytes, HostPipe** hp,
              const float** src) {
    *hp = nullptr;
    *src = (const float*)dev;
    int rc;
    if (bytes + result_bytes < kHostPipeBytes) {
        if ((rc = ensure_host(c, c->hx, bytes)) != SMX_OK) return rc;
        std::memcpy(c->hx.p, host, bytes);
        if (read_once) {
            *src = (const float*)c->hx.p;
            return SMX_OK;
        }
        return staged_to_device(c, dev, c->hx.p, bytes);
    }
    if (!(*hp = host_pipe(c))) {
        SMX_HIP(c, hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, c->stream));
        return SMX_OK;
    }
    rc = (*hp)->begin(c);
    if (rc == SMX_OK) rc = (*hp)->in(c, dev, host, bytes);
    if (rc == SMX_OK) rc = (*hp)->in_done(c);
    if (rc != SMX_OK) return (*hp)->end(c, rc);
    (*hp)->populate(result, result_bytes);
    return SMX_OK;
}

int host_receive(smx_ctx* c, void* host, const void* dev, size_t bytes, HostPipe* hp, int rc) {
    if (hp) {
        if (rc == SMX_OK) rc = hp->out(c, host, dev, bytes);
        return hp->end(c, rc);
    }
    HostCall call(c);
    if (rc != SMX_OK) return rc;
    if (bytes >= kHostPipeBytes) {   // (no pipe)
        SMX_HIP(c, hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, c->stream));
        SMX_HIP(c, hipStreamSynchronize(c->stream));
        return call.done();
    }
    // The result crosses as parts that report themselves (span_out_kernel), each copied on while the next ones are on the
    // bus.  (A copy command and a wait: the wait alone is 8 us dearer behind a copy than behind a kernel.)
    constexpr size_t kPart = HostPipe::kPart;
    static_assert(kHostPipeBytes / kPart + 1 <= kHostFlags - 64, "one report word per part");
    if ((rc = ensure_host(c, c->hy, bytes)) != SMX_OK) return rc;
    const unsigned parts = (unsigned)((bytes + kPart - 1) / kPart), want = ++c->flag_seq;
    hipLaunchKernelGGL(span_out_kernel, dim3(std::min(parts, HostPipe::kOutWgs)), dim3(256), 0, c->stream, (const char*)dev, c->hy.p, bytes,
                       c->hflag + 64, want);
    SMX_HIP(c, hipGetLastError());
    const volatile unsigned* flag = c->hflag + 64;
    const auto t0 = std::chrono::steady_clock::now();
    unsigned p = 0;
    for (unsigned i = 1; p < parts; i++) {
        unsigned q = p;
        while (q < parts && flag[q] == want) q++;
        if (q > p) {
            std::atomic_thread_fence(std::memory_order_acquire);
            const size_t o = p * kPart, e = std::min<size_t>(q * kPart, bytes);
            std::memcpy((char*)host + o, c->hy.p + o, e - o);
            p = q;
            continue;
        }
        __builtin_ia32_pause();
        if (i % 64 == 0 && std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count() > 2.0) {   // long work, or a failed launch
            SMX_HIP(c, hipStreamSynchronize(c->stream));
            std::memcpy((char*)host + p * kPart, c->hy.p + p * kPart, bytes - p * kPart);
            break;
        }
    }
    return call.done();
}

HostPipe* host_pipe(smx_ctx* c) {
    if (c->pipe || c->pipe_refused) return c->pipe;
    HostPipe* p = new (std::nothrow) HostPipe();
    int rc = SMX_ERR_NOMEM;
    try {
        if (p) rc = p->open(c);
    } catch (const std::exception&) {   // out of host memory
    }
    if (rc == SMX_OK) c->pipe = p;
    else delete p;
    c->pipe_refused = rc != SMX_OK;
    return c->pipe;
}

}  // namespace smx
