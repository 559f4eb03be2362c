// Test double of the HIP runtime functions that libstrix_mi355.so calls, for its host side on a machine without a GPU: memory
// is malloc'ed, every stream is a thread that runs its commands in order, and of the kernels only those that move bytes or
// report to the host do anything.  Fresh device memory holds word i = i, so that a result copied out of memory no kernel has
// written tells where it comes from; allocations and copies of more than a gigabyte are not filled or made.
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

struct ihipStream_t {
    std::mutex mu;
    std::condition_variable cv;
    std::deque<std::function<void()>> queue;
    size_t enqueued = 0, completed = 0;
    bool quit = false, capturing = false, broken = false;
    std::thread thread;
    ihipStream_t() : thread([this] { run(); }) {}
    ~ihipStream_t() {
        {
            std::lock_guard<std::mutex> l(mu);
            quit = true;
        }
        cv.notify_all();
        thread.join();
    }
    void run() {
        std::unique_lock<std::mutex> l(mu);
        for (;;) {
            cv.wait(l, [&] { return quit || !queue.empty(); });
            if (queue.empty()) return;
            auto f = std::move(queue.front());
            queue.pop_front();
            l.unlock();
            f();
            l.lock();
            completed++;
            cv.notify_all();
        }
    }
    void add(std::function<void()> f) {
        if (capturing) return;   // recorded, not run
        {
            std::lock_guard<std::mutex> l(mu);
            queue.push_back(std::move(f));
            enqueued++;
        }
        cv.notify_all();
    }
    void drain() {
        std::unique_lock<std::mutex> l(mu);
        const size_t want = enqueued;
        cv.wait(l, [&] { return completed >= want; });
    }
};
struct Mark {   // one recording of an event
    std::mutex mu;
    std::condition_variable cv;
    bool done = false;
    void wait() {
        std::unique_lock<std::mutex> l(mu);
        cv.wait(l, [&] { return done; });
    }
    void set() {
        std::lock_guard<std::mutex> l(mu);
        done = true;
        cv.notify_all();
    }
};
struct ihipEvent_t {
    std::shared_ptr<Mark> mark;
    bool in_capture = false;
};

namespace {
constexpr size_t kGigabyte = size_t(1) << 30;
std::mutex g_mu;
std::map<const void*, std::string> g_kernels;
std::vector<ihipStream_t*> g_streams;
std::string g_inbound, g_slow_kernel, g_failing_kernel;
bool g_keep_inbound = false;
int g_slow_us = 0;
size_t g_host_limit = SIZE_MAX, g_host_live = 0;
std::map<void*, size_t> g_host;
std::atomic<int> g_host_refused{0}, g_launches{0}, g_failed_launches{0};
std::vector<unsigned> g_host_flags;
thread_local hipError_t t_last = hipSuccess;
struct Config { dim3 grid, block; size_t shmem; hipStream_t stream; };
thread_local Config t_config;
alignas(256) char g_symbol[1 << 20];

hipError_t done(hipError_t e) {
    if (e != hipSuccess) t_last = e;
    return e;
}
template <class T>
T arg(void** args, int i) {
    T v;
    std::memcpy(&v, args[i], sizeof v);
    return v;
}
}  // namespace

extern "C" {

// ---- what the tests set and ask ----
void fake_keep_inbound(int on) {
    std::lock_guard<std::mutex> l(g_mu);
    g_keep_inbound = on != 0;
    g_inbound.clear();
}
size_t fake_inbound(char* out, size_t cap) {   // what host-to-device copy commands have carried, in order
    std::lock_guard<std::mutex> l(g_mu);
    std::memcpy(out, g_inbound.data(), std::min(cap, g_inbound.size()));
    return g_inbound.size();
}
void fake_host_limit(size_t bytes) { g_host_limit = bytes; }   // a larger pinned allocation is refused
int fake_host_refused() { return g_host_refused; }
size_t fake_host_live() { return g_host_live; }
int fake_host_noncoherent() {   // pinned allocations that did not ask for coherent memory
    std::lock_guard<std::mutex> l(g_mu);
    int n = 0;
    for (unsigned f : g_host_flags) n += (f & hipHostMallocCoherent) == 0;
    return n;
}
void fake_slow_kernel(const char* name, int us) {
    std::lock_guard<std::mutex> l(g_mu);
    g_slow_kernel = name;
    g_slow_us = us;
}
void fake_failing_kernel(const char* name) {   // launches of it fail
    std::lock_guard<std::mutex> l(g_mu);
    g_failing_kernel = name;
}
int fake_failed_launches() { return g_failed_launches; }
int fake_launches() { return g_launches; }
size_t fake_pending() {   // commands that have been enqueued and have not finished
    std::lock_guard<std::mutex> l(g_mu);
    size_t n = 0;
    for (auto* s : g_streams) {
        std::lock_guard<std::mutex> k(s->mu);
        n += s->enqueued - s->completed;
    }
    return n;
}
int fake_streams() {
    std::lock_guard<std::mutex> l(g_mu);
    return (int)g_streams.size();
}

// ---- registration and launch ----
void** __hipRegisterFatBinary(const void*) {
    static void* h;
    return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { g_kernels[host] = name; }
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, hipStream_t stream) {
    t_config = {grid, block, shmem, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shmem, hipStream_t* stream) {
    *grid = t_config.grid; *block = t_config.block; *shmem = t_config.shmem; *stream = t_config.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t s) {
    std::string name;
    int us = 0;
    {
        std::lock_guard<std::mutex> l(g_mu);
        name = g_kernels[f];
        if (!g_failing_kernel.empty() && name.find(g_failing_kernel) != std::string::npos) {
            g_failed_launches++;
            return done(hipErrorLaunchFailure);
        }
        if (!g_slow_kernel.empty() && name.find(g_slow_kernel) != std::string::npos) us = g_slow_us;
    }
    g_launches++;
    const auto is = [&](const char* n) { return name.find(n) != std::string::npos; };
    std::function<void()> body = [] {};
    if (is("span_out_kernel")) {
        auto src = arg<const char*>(args, 0);
        auto dst = arg<char*>(args, 1);
        auto n = arg<size_t>(args, 2);
        auto flags = arg<unsigned*>(args, 3);
        auto seq = arg<unsigned>(args, 4);
        body = [=] {
            for (size_t o = 0, p = 0; o < n; o += 16384, p++) {
                std::memcpy(dst + o, src + o, std::min<size_t>(16384, n - o));
                __atomic_store_n(flags + p, seq, __ATOMIC_RELEASE);
            }
        };
    } else if (is("span_in_kernel")) {
        auto src = arg<const char*>(args, 0);
        auto dst = arg<char*>(args, 1);
        auto n = arg<size_t>(args, 2);
        body = [=] { std::memcpy(dst, src, n * 4); };
    } else if (is("stream_flag_kernel")) {
        auto flag = arg<unsigned*>(args, 0);
        auto value = arg<unsigned>(args, 1);
        body = [=] { __atomic_store_n(flag, value, __ATOMIC_RELEASE); };
    }
    s->add([us, body] {
        if (us) std::this_thread::sleep_for(std::chrono::microseconds(us));
        body();
    });
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) {
    *p = g_symbol;
    return hipSuccess;
}

// ---- device, errors ----
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->name, "test double");
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = t_last;
    t_last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "an error of the test double"; }

// ---- memory ----
hipError_t hipMalloc(void** p, size_t n) {
    const size_t words = (n + 3) / 4;
    unsigned* w = (unsigned*)std::aligned_alloc(4096, (words * 4 + 4095) & ~size_t(4095));
    if (!w) return done(hipErrorOutOfMemory);
    for (size_t i = 0; n <= kGigabyte && i < words; i++) w[i] = (unsigned)i;
    *p = w;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned flags) {
    if (n > g_host_limit) {
        g_host_refused++;
        return done(hipErrorOutOfMemory);
    }
    *p = std::aligned_alloc(4096, (n + 4095) & ~size_t(4095));
    std::memset(*p, 0xee, n);
    std::lock_guard<std::mutex> l(g_mu);
    g_host[*p] = n;
    g_host_live += n;
    g_host_flags.push_back(flags);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::lock_guard<std::mutex> l(g_mu);
    g_host_live -= g_host[p];
    g_host.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind kind, hipStream_t s) {
    bool pinned;
    {
        std::lock_guard<std::mutex> l(g_mu);
        const auto in = [&](const void* p) {
            auto it = g_host.upper_bound((void*)p);
            return it != g_host.begin() && (--it, (const char*)p < (const char*)it->first + it->second);
        };
        pinned = in(src) || in(dst);
    }
    s->add([=] {
        if (n <= kGigabyte) std::memcpy(dst, src, n);
        if (kind == hipMemcpyHostToDevice) {
            std::lock_guard<std::mutex> l(g_mu);
            if (g_keep_inbound && n <= kGigabyte) g_inbound.append((const char*)dst, n);
        }
    });
    if (!pinned && kind == hipMemcpyHostToDevice && !s->capturing) s->drain();   // pageable memory: staged before the call returns
    return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void* dst, size_t dp, const void* src, size_t sp, size_t w, size_t h, hipMemcpyKind, hipStream_t s) {
    s->add([=] {
        for (size_t i = 0; i < h; i++) std::memcpy((char*)dst + i * dp, (const char*)src + i * sp, w);
    });
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t s) {
    s->add([=] { std::memset(p, v, n); });
    return hipSuccess;
}

// ---- streams, events, graphs ----
hipError_t hipStreamCreate(hipStream_t* s) {
    *s = new ihipStream_t();
    std::lock_guard<std::mutex> l(g_mu);
    g_streams.push_back(*s);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return hipStreamCreate(s); }
hipError_t hipStreamDestroy(hipStream_t s) {
    {
        std::lock_guard<std::mutex> l(g_mu);
        for (auto it = g_streams.begin(); it != g_streams.end(); ++it)
            if (*it == s) {
                g_streams.erase(it);
                break;
            }
    }
    s->drain();
    delete s;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    if (s->capturing) {
        s->broken = true;
        return done(hipErrorStreamCaptureUnsupported);
    }
    s->drain();
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = new ihipEvent_t();
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) {
    delete e;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    auto m = std::make_shared<Mark>();
    e->mark = m;
    e->in_capture = s->capturing;
    s->add([m] { m->set(); });
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) {
    if (!e->mark) return hipSuccess;
    std::lock_guard<std::mutex> l(e->mark->mu);
    return e->mark->done ? hipSuccess : done(hipErrorNotReady);
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    if (e->in_capture) return done(hipErrorCapturedEvent);
    if (e->mark) e->mark->wait();
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 0;
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    if (e->in_capture) {   // the waiting stream joins the capture
        s->capturing = true;
        return hipSuccess;
    }
    if (auto m = e->mark) s->add([m] { m->wait(); });
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
    s->capturing = true;
    s->broken = false;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
    s->capturing = false;
    *g = nullptr;
    return s->broken ? done(hipErrorStreamCaptureInvalidated) : hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    *x = nullptr;
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

}  // extern "C"
