// A stand-in for the HIP runtime that runs nothing and writes down what it is asked for, so that the host side of the
// library can be tested without a GPU: the order of launches over streams and events, and what happens when a call fails.
// Loaded before the library with its symbols global (tests/test_host_failures_cpu.py).
//
// Log lines:  launch <kernel> <stream> | record <event> <stream> | wait <stream> <event> | graph - <stream>
// Streams and events are numbered; the default stream is 0.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <new>
#include <set>
#include <string>

namespace {

struct Stream {
    bool capturing = false;
    Stream* origin = nullptr;   // of the capture it takes part in
    std::set<Stream*> open;     // (origin) streams with captured work that no other stream has waited for
    long ops = 0;               // launches and waits so far
    void did() {
        ++ops;
        if (capturing && origin != this) origin->open.insert(this);
    }
};
struct Event {
    int id;
    Stream* on = nullptr;
    bool captured = false;
    long at = 0;  // of on->ops
};

std::string& log_text() {
    static std::string s;
    return s;
}
long fail_new = -1;  // calls of operator new until they fail
struct Own {  // what this file allocates itself does not count
    const long keep = fail_new;
    Own() { fail_new = -1; }
    ~Own() { fail_new = keep; }
};
std::map<const void*, std::string>& kernels() {
    static std::map<const void*, std::string> m;
    return m;
}
Stream& default_stream() {
    static Stream s;
    return s;
}
std::map<Stream*, int>& streams() {
    static std::map<Stream*, int> m;
    return m;
}
Stream* stream_of(hipStream_t s) { return s ? reinterpret_cast<Stream*>(s) : &default_stream(); }
int number(Stream* s) { return s == &default_stream() ? 0 : streams()[s]; }
void note(const char* what, const char* name, int number) {
    Own own;
    log_text() += std::string(what) + " " + name + " " + std::to_string(number) + "\n";
}
void note(const char* what, int a, int b) {
    Own own;
    note(what, std::to_string(a).c_str(), b);
}

hipError_t last_error = hipSuccess;
long launches = 0, fail_from = -1, fail_to = -1;     // launches that report an error
unsigned long long largest_allocation = ~0ull;
int next_event = 0;

hipError_t report(hipError_t e) {
    if (e != hipSuccess) last_error = e;
    return e;
}

}  // namespace

// every operator new of the library
void* operator new(std::size_t n) {
    if (fail_new == 0) throw std::bad_alloc();
    if (fail_new > 0) --fail_new;
    void* p = std::malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

extern "C" {

const char* fake_log() { return log_text().c_str(); }
void fake_clear_log() { log_text().clear(); }
void fake_fail_launches(long first, long count) {  // counted from the next one
    fail_from = first < 0 ? -1 : launches + first;
    fail_to = fail_from + count;
}
void fake_largest_allocation(unsigned long long bytes) { largest_allocation = bytes; }
void fake_fail_new(long after) { fail_new = after; }  // (a negative number: never again)
long fake_news_left() { return fail_new; }
int fake_stream_number(hipStream_t s) { return number(stream_of(s)); }

void** __hipRegisterFatBinary(const void*) {
    static void* handle = nullptr;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned int, void*, void*, dim3*, dim3*, int*) {
    kernels()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
struct {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
} pushed;
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream) {
    pushed = {grid, block, lds, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream) {
    *grid = pushed.grid;
    *block = pushed.block;
    *lds = pushed.lds;
    *stream = pushed.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void**, size_t, hipStream_t s) {
    if (grid.x == 0) return report(hipErrorInvalidConfiguration);
    note("launch", kernels()[f].c_str(), number(stream_of(s)));
    Own own;
    stream_of(s)->did();
    const long i = launches++;
    if (fail_from >= 0 && i >= fail_from && i < fail_to) return report(hipErrorUnknown);
    return hipSuccess;
}

hipError_t hipGetLastError() {
    const hipError_t e = last_error;
    last_error = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "made to fail"; }
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
    *v = 256;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void**, const void*) { return report(hipErrorInvalidSymbol); }

hipError_t hipMalloc(void** p, size_t n) {
    *p = nullptr;
    if (n > largest_allocation) return report(hipErrorOutOfMemory);
    *p = std::aligned_alloc(256, (n + 255) / 256 * 256);
    return *p ? hipSuccess : report(hipErrorOutOfMemory);
}
hipError_t hipFree(void* p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned int) {
    Stream* st = new Stream();
    const int id = (int)streams().size() + 1;
    streams()[st] = id;
    *s = reinterpret_cast<hipStream_t>(st);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* c) {
    *c = stream_of(s)->capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
    Stream* st = stream_of(s);
    if (st->capturing || !s) return report(hipErrorIllegalState);
    st->capturing = true;
    st->origin = st;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
    Stream* st = stream_of(s);
    *g = nullptr;
    if (!st->capturing) return report(hipErrorIllegalState);
    const bool open = !st->open.empty();
    for (auto& other : streams())
        if (other.first->origin == st) {
            other.first->capturing = false;
            other.first->origin = nullptr;
        }
    st->open.clear();
    if (open) return report(hipErrorStreamCaptureUnjoined);
    *g = reinterpret_cast<hipGraph_t>(&default_stream());  // (only compared with null)
    return hipSuccess;
}

hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    Own own;
    Event* ev = new Event();
    ev->id = next_event++;
    *e = reinterpret_cast<hipEvent_t>(ev);
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) {
    delete reinterpret_cast<Event*>(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    Event* ev = reinterpret_cast<Event*>(e);
    ev->on = stream_of(s);
    ev->captured = ev->on->capturing;
    ev->at = ev->on->ops;
    note("record", ev->id, number(ev->on));
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned int) {
    Own own;
    Event* ev = reinterpret_cast<Event*>(e);
    Stream* st = stream_of(s);
    if (!ev->on) return hipSuccess;
    if (ev->captured && ev->on->capturing) {
        if (!st->capturing) {  // a fork
            st->capturing = true;
            st->origin = ev->on->origin;
        }
        if (ev->at == ev->on->ops) st->origin->open.erase(ev->on);
        st->did();
    } else if (st->capturing) {
        return report(hipErrorStreamCaptureIsolation);
    }
    note("wait", number(st), ev->id);
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 0.f;
    return hipSuccess;
}

hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
    *x = reinterpret_cast<hipGraphExec_t>(g);
    return hipSuccess;
}
hipError_t hipGraphGetNodes(hipGraph_t, hipGraphNode_t*, size_t* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t s) {
    note("graph", "-", number(stream_of(s)));
    const long i = launches++;
    if (fail_from >= 0 && i >= fail_from && i < fail_to) return report(hipErrorUnknown);
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }

}  // extern "C"
