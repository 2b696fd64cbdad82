// A HIP runtime on the CPU for tests of the library's host code: device memory
// is host memory, and work queued on a stream runs only when the host waits for
// that stream, an event of it, or the device (hipFree), which is the latest a
// device may run it. The default stream is one more queue: the library's streams
// are non-blocking and order nothing against it. Errors stay until
// hipGetLastError reads them. Of the kernels only the quantizer computes
// (fh_quantize); launches of others are dropped. fake_fail(name, n) makes the
// n-th next call of an allocation or creation fail.
#include <dlfcn.h>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <set>
#include <string>

struct Dim3 {
    uint32_t x, y, z;
};
struct Stream {
    std::deque<std::function<void()>> queue;
};
struct Event {
    Stream* stream = nullptr;
};

static std::recursive_mutex mu;
static Stream default_stream;
static std::set<Stream*> streams;
static std::map<const void*, std::string> kernels;
static std::map<std::string, int> failures;
static thread_local int last_error;
static int launched, waits, widest, pinned;

using Lock = std::lock_guard<std::recursive_mutex>;

static void drain(Stream* s) {
    while (!s->queue.empty()) {
        auto f = std::move(s->queue.front());
        s->queue.pop_front();
        f();
    }
}
static Stream* of(void* s) { return s ? (Stream*)s : &default_stream; }
static int error(int e) { return last_error = e; }
static bool fails(const char* name) {
    auto it = failures.find(name);
    return it != failures.end() && it->second > 0 && --it->second == 0;
}

extern "C" {

void fake_fail(const char* name, int nth) {
    Lock l(mu);
    failures[name] = nth;
}
int fake_pending_default() {
    Lock l(mu);
    return (int)default_stream.queue.size();
}
int fake_launched() { return launched; }
int fake_waits() { return waits; }
int fake_pinned() { return pinned; }  // pinned allocations
int fake_widest() { return widest; }  // the largest grid y of a launch

void** __hipRegisterFatBinary(const void*) {
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*,
                           int*) {
    kernels[host] = name;
}
static thread_local struct {
    Dim3 grid, block;
    size_t shared;
    void* stream;
} call;
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shared, void* stream) {
    call = {grid, block, shared, stream};
    return 0;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* shared, void** stream) {
    *grid = call.grid;
    *block = call.block;
    *shared = call.shared;
    *stream = call.stream;
    return 0;
}

int hipLaunchKernel(const void* f, Dim3 grid, Dim3, void** a, size_t, void* stream) {
    Lock l(mu);
    launched++;
    if ((int)grid.y > widest) widest = grid.y;
    const std::string name = kernels[f];
    const size_t at = name.find("k_quantizeILb");
    if (at == std::string::npos) return 0;
    // (w, cs, imp, cols, q, qt, s): a call without cs and qt is fh_quantize's, the search's others are dropped
    const float *w = *(const float**)a[0], *cs = *(const float**)a[1], *imp = *(const float**)a[2];
    const int cols = *(int*)a[3], kind = name[at + 13] == '1' ? 1 : 2;
    uint8_t* q = *(uint8_t**)a[4];
    float* s = *(float**)a[6];
    if (cs || *(void**)a[5]) return 0;
    using Quantize = int (*)(int, int, int, const float*, const float*, uint8_t*, float*);
    static const Quantize quantize = (Quantize)dlsym(dlopen(getenv("FERRO_GPU_LIB"), RTLD_NOW), "fh_quantize");
    of(stream)->queue.push_back([=] { quantize(kind, (int)grid.x * 32, cols, w, imp, q, s); });
    return 0;
}
int hipExtLaunchKernel(const void*, Dim3, Dim3, void**, size_t, void*, void*, void*, int) {
    launched++;
    return 0;
}

int hipGetDeviceCount(int* n) {
    *n = 1;
    return 0;
}
int hipSetDevice(int) { return 0; }
const char* hipGetErrorString(int) { return "fake error"; }
int hipGetLastError() {
    const int e = last_error;
    last_error = 0;
    return e;
}

static int make(void** p, size_t n, const char* name) {
    Lock l(mu);
    // (sizes beyond any card's memory fail as there)
    if (fails(name) || n > (size_t)1 << 38 || !(*p = malloc(n))) return error(2);
    memset(*p, 0xA5, n < 4096 ? n : 4096);
    return 0;
}
int hipMalloc(void** p, size_t n) { return make(p, n, "hipMalloc"); }
int hipHostMalloc(void** p, size_t n, unsigned) {
    pinned++;
    return make(p, n, "hipHostMalloc");
}
int hipFree(void* p) {
    Lock l(mu);
    drain(&default_stream);
    for (Stream* s : streams) drain(s);
    free(p);
    return 0;
}
int hipHostFree(void* p) { return hipFree(p); }
int hipGetSymbolAddress(void** p, const void* host) {
    static std::map<const void*, void*> at;
    Lock l(mu);
    if (!at[host]) at[host] = calloc(1, (size_t)4 << 20);
    *p = at[host];
    return 0;
}

int hipStreamCreateWithFlags(void** s, unsigned) {
    Lock l(mu);
    if (fails("hipStreamCreateWithFlags")) return error(2);
    Stream* n = new Stream();
    streams.insert(n);
    *s = n;
    return 0;
}
int hipStreamSynchronize(void* s) {
    Lock l(mu);
    waits++;
    drain(of(s));
    return 0;
}
int hipStreamDestroy(void* s) {
    Lock l(mu);
    drain(of(s));
    streams.erase((Stream*)s);
    delete (Stream*)s;
    return 0;
}
int hipEventCreate(void** e) {
    if (fails("hipEventCreate")) return error(2);
    *e = new Event();
    return 0;
}
int hipEventCreateWithFlags(void** e, unsigned) {
    Lock l(mu);
    if (fails("hipEventCreateWithFlags")) return error(2);
    *e = new Event();
    return 0;
}
int hipEventDestroy(void* e) {
    delete (Event*)e;
    return 0;
}
int hipEventRecord(void* e, void* s) {
    ((Event*)e)->stream = of(s);
    return 0;
}
int hipEventSynchronize(void* e) {
    Lock l(mu);
    if (((Event*)e)->stream) drain(((Event*)e)->stream);
    return 0;
}
int hipEventElapsedTime(float* ms, void*, void*) {
    *ms = 0.0f;
    return 0;
}

int hipMemset(void* p, int v, size_t n) {
    Lock l(mu);
    default_stream.queue.push_back([=] { memset(p, v, n); });
    return 0;
}
int hipMemsetAsync(void* p, int v, size_t n, void* s) {
    Lock l(mu);
    if (fails("hipMemsetAsync")) return error(1);
    of(s)->queue.push_back([=] { memset(p, v, n); });
    return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int) {
    Lock l(mu);
    drain(&default_stream);
    memcpy(d, s, n);
    return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void* st) {
    Lock l(mu);
    of(st)->queue.push_back([=] { memcpy(d, s, n); });
    return 0;
}

// (step graphs are not taken here)
int hipStreamBeginCapture(void*, int) { return error(801); }
int hipStreamEndCapture(void*, void**) { return error(801); }
int hipGraphInstantiate(void**, void*, void*, char*, size_t) { return error(801); }
int hipGraphLaunch(void*, void*) { return error(801); }
int hipGraphDestroy(void*) { return 0; }
int hipGraphExecDestroy(void*) { return 0; }
}
