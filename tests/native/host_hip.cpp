// A stand-in on the CPU for the HIP calls that the library's host code makes,
// so that its threads, pools, staging and captures can be driven without a GPU.
// Device memory is host memory.  Every stream is a thread that takes its
// operations in order; events, captures and graphs follow the streams.  Of the
// kernels only the one that writes a mode's map does anything (host_hip.h).
#include <hip/hip_runtime.h>

#include <sys/mman.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <memory>
#include <mutex>
#include <set>
#include <string>
#include <thread>
#include <vector>

#include "../../sister_amd/csrc/rig.h"
#include "host_hip.h"

namespace host_hip {
std::atomic<long> pinned_bytes{0};
std::atomic<int> branches{0}, captures{0}, step_us{0};
std::atomic<size_t> device_bytes{(size_t)64 << 30};
}  // namespace host_hip
using namespace host_hip;

namespace {

typedef std::function<void()> Op;

[[noreturn]] void die(const char* what)
{
    std::printf("host_hip: %s\n", what);
    std::fflush(stdout);
    std::_Exit(3);
}

struct Capture;
struct Stream {
    std::mutex mu;
    std::condition_variable cv;
    std::deque<Op> ops;
    bool busy = false, stop = false;
    Capture* cap = nullptr;      // the capture this stream records into
    std::thread th;
    Stream()
    {
        th = std::thread([this] {
            std::unique_lock<std::mutex> lk(mu);
            for (;;) {
                cv.wait(lk, [&] { return stop || !ops.empty(); });
                if (ops.empty()) return;
                Op op = std::move(ops.front());
                ops.pop_front();
                busy = true;
                lk.unlock();
                op();
                lk.lock();
                busy = false;
                cv.notify_all();
            }
        });
    }
    void push(Op op)
    {
        std::lock_guard<std::mutex> lk(mu);
        ops.push_back(std::move(op));
        cv.notify_all();
    }
    void drain()
    {
        std::unique_lock<std::mutex> lk(mu);
        cv.wait(lk, [&] { return ops.empty() && !busy; });
    }
    ~Stream()
    {
        drain();
        {
            std::lock_guard<std::mutex> lk(mu);
            stop = true;
            cv.notify_all();
        }
        th.join();
    }
};
// operations in the order they were recorded (an order that its events allow)
struct Capture {
    Stream* origin;
    std::vector<Op> ops;
    std::set<Stream*> joined, open;   // streams that take part; those with work not waited for
};
struct Event {
    std::mutex mu;
    std::condition_variable cv;
    long asked = 0, done = 0;
    Capture* cap = nullptr;           // recorded inside this capture
    Stream* from = nullptr;
};

// kernels are registered before this file's own variables are set up
std::map<const void*, std::string>& kernels()
{
    static std::map<const void*, std::string> m;
    return m;
}
std::mutex g_mu;
std::map<void*, size_t> g_dev, g_pin;
Stream* S(hipStream_t s) { return (Stream*)s; }
Event* E(hipEvent_t e) { return (Event*)e; }

void issue(Stream* s, Op op)
{
    if (s->cap) {
        s->cap->open.insert(s);
        s->cap->ops.push_back(std::move(op));
    } else {
        s->push(std::move(op));
    }
}

void* map_bytes(size_t n)
{
    void* p = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    return p == MAP_FAILED ? nullptr : p;
}
hipError_t drop(std::map<void*, size_t>& m, void* p, bool pin)
{
    if (!p) return hipSuccess;
    std::lock_guard<std::mutex> lk(g_mu);
    auto it = m.find(p);
    if (it == m.end()) die("a free of memory that is not held");
    munmap(p, it->second);
    if (pin) pinned_bytes -= (long)it->second;
    m.erase(it);
    return hipSuccess;
}

struct Config { dim3 grid, block; size_t lds; hipStream_t st; };
thread_local std::vector<Config> t_config;

}  // namespace

extern "C" {

void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char* dev, const char*, unsigned, void*, void*, void*, void*, int*)
{
    kernels()[f] = dev;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t st)
{
    t_config.push_back({g, b, lds, st});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* st)
{
    const Config c = t_config.back();
    t_config.pop_back();
    *g = c.grid; *b = c.block; *lds = c.lds; *st = c.st;
    return hipSuccess;
}

hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t st)
{
    const std::string& name = kernels().at(f);
    if (name.find("k_winner") == std::string::npos) {
        issue(S(st), [] { std::this_thread::sleep_for(std::chrono::microseconds(step_us)); });
        return hipSuccess;
    }
    const auto* rigs = *(const sister::RigDesc**)args[0];
    const int n = *(int*)args[1], mode = *(int*)args[3];
    issue(S(st), [=] {
        for (int k = 0; k < n; k++) {
            const sister::RigDesc& g = rigs[k];
            for (int y = 0; y < g.H; y++)
                for (int x = 0; x < g.W; x++) {
                    int v = 0;
                    for (int i = 0; i < 5; i++) v += (i + 1) * g.view[i][(size_t)y * g.stride + x];
                    const size_t o = (size_t)y * g.W + x;
                    if (g.out[mode]) g.out[mode][o] = (uint16_t)map_value(v, mode);
                    if (mode == 0 && g.disp) g.disp[o] = (uint16_t)v;
                    if (mode == 0 && g.subpix) g.subpix[o] = (float)v;
                }
        }
    });
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*)
{
    static void* scratch = map_bytes((size_t)256 << 20);
    *p = scratch;
    return hipSuccess;
}

hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int)
{
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 160 << 10;
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) { *f = *t = device_bytes; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "error"; }

hipError_t hipMalloc(void** p, size_t n)
{
    *p = map_bytes(n);
    if (!*p) return hipErrorOutOfMemory;
    std::lock_guard<std::mutex> lk(g_mu);
    g_dev[*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void* p) { return drop(g_dev, p, false); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    *p = map_bytes(n);
    if (!*p) return hipErrorOutOfMemory;
    std::lock_guard<std::mutex> lk(g_mu);
    g_pin[*p] = n;
    pinned_bytes += (long)n;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) { return drop(g_pin, p, true); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st)
{
    issue(S(st), [=] {
        std::this_thread::sleep_for(std::chrono::microseconds(step_us));
        std::memcpy(d, s, n);
    });
    return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, hipMemcpyKind, hipStream_t st)
{
    issue(S(st), [=] {
        for (size_t y = 0; y < h; y++) std::memcpy((char*)d + y * dp, (const char*)s + y * sp, w);
    });
    return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t) new Stream; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { delete S(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s)
{
    if (S(s)->cap) die("a wait for a stream that is being captured");
    S(s)->drain();
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t st, hipEvent_t ev, unsigned)
{
    Stream* s = S(st);
    Event* e = E(ev);
    if (e->cap) {   // fork or join of a capture
        if (s->cap && s->cap != e->cap) die("an event of another capture");
        if (!s->cap) {
            s->drain();
            s->cap = e->cap;
            s->cap->joined.insert(s);
        }
        e->cap->open.erase(e->from);
        e->cap->open.insert(s);
        return hipSuccess;
    }
    if (s->cap) die("a captured stream waits for an event outside the capture");
    long want;
    {
        std::lock_guard<std::mutex> lk(e->mu);
        want = e->asked;
    }
    s->push([=] {
        std::unique_lock<std::mutex> lk(e->mu);
        e->cv.wait(lk, [&] { return e->done >= want; });
    });
    return hipSuccess;
}

hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t) new Event; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { delete E(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t ev, hipStream_t st)
{
    Event* e = E(ev);
    Stream* s = S(st);
    e->cap = s->cap;
    e->from = s;
    if (s->cap) return hipSuccess;
    long mine;
    {
        std::lock_guard<std::mutex> lk(e->mu);
        mine = ++e->asked;
    }
    s->push([=] {
        std::lock_guard<std::mutex> lk(e->mu);
        if (mine > e->done) e->done = mine;
        e->cv.notify_all();
    });
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t ev)
{
    Event* e = E(ev);
    if (e->cap) die("a wait for an event of a capture");
    std::unique_lock<std::mutex> lk(e->mu);
    const long want = e->asked;
    e->cv.wait(lk, [&] { return e->done >= want; });
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t ev)
{
    Event* e = E(ev);
    std::lock_guard<std::mutex> lk(e->mu);
    return e->done >= e->asked ? hipSuccess : hipErrorNotReady;
}
hipError_t hipEventElapsedTime(float* t, hipEvent_t, hipEvent_t) { *t = 0; return hipSuccess; }

hipError_t hipStreamBeginCapture(hipStream_t st, hipStreamCaptureMode)
{
    Stream* s = S(st);
    if (s->cap) die("a stream is captured twice");
    s->cap = new Capture{s, {}, {}, {}};
    captures++;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t st, hipGraph_t* g)
{
    Stream* s = S(st);
    Capture* c = s->cap;
    if (!c || c->origin != s) die("the end of a capture that was not begun");
    c->open.erase(s);
    if (!c->open.empty()) die("a capture ends with a stream that was not joined");
    for (Stream* j : c->joined) j->cap = nullptr;
    s->cap = nullptr;
    const int n = (int)c->joined.size() + 1;
    if (n > branches) branches = n;
    *g = (hipGraph_t)c;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t g, hipGraphNode_t*, char*, size_t)
{
    *x = (hipGraphExec_t) new std::vector<Op>(((Capture*)g)->ops);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t st)
{
    for (const Op& op : *(std::vector<Op>*)x) issue(S(st), op);
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { delete (std::vector<Op>*)x; return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { delete (Capture*)g; return hipSuccess; }

}  // extern "C"
