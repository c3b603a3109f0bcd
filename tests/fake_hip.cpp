// fake_hip.cpp -- a stand-in for the HIP runtime on the CPU, for tests of the
// library's host code: device memory is host memory, kernels are recorded and
// (but for the field reads below) not run.  It checks nothing that kernels
// compute; it shows what the host code allocates, on which device, what it
// captures, and what it does when a call fails.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

namespace {

struct Object {
    int device;
};

std::mutex lock;
std::map<std::string, long long> counters;
std::map<const void*, std::string> kernels;
std::map<void*, size_t> sizes;
std::map<std::string, long long> fail_from;   // call -> number of calls that still succeed
thread_local int current = 0;
thread_local int last_error = 0;
size_t free_bytes = (size_t)1 << 38;
int wrong_device = 0;   // uses of an object on another device's stream

int err(int e) {
    if (e) last_error = e;
    return e;
}

bool fails(const char* name) {
    auto it = fail_from.find(name);
    return it != fail_from.end() && it->second-- <= 0;
}

void count(const std::string& name, long long v = 1) {
    std::lock_guard<std::mutex> g(lock);
    counters[name] += v;
}

std::string on_device(const char* what) { return std::string(what) + "@" + std::to_string(current); }

}  // namespace

extern "C" {

// ---- the tests' side ----
long long fake_count(const char* name) {
    std::lock_guard<std::mutex> g(lock);
    return counters[name];
}
// launches of the kernels whose mangled names hold `part`
long long fake_launches(const char* part) {
    std::lock_guard<std::mutex> g(lock);
    long long n = 0;
    for (auto& c : counters)
        if (c.first.compare(0, 8, "mangled ") == 0 && c.first.find(part) != std::string::npos) n += c.second;
    return n;
}
void fake_fail(const char* name, long long after) { fail_from[name] = after; }
void fake_work(const char* name) { fail_from.erase(name); }
void fake_free_bytes(size_t n) { free_bytes = n; }
int fake_wrong_device() { return wrong_device; }
int fake_set_device(int d) {
    current = d;
    return 0;
}
int fake_get_device() { return current; }

// ---- devices, errors ----
int hipGetDeviceCount(int* n) {
    *n = 2;
    return 0;
}
int hipGetDevice(int* d) {
    *d = current;
    return 0;
}
int hipSetDevice(int d) {
    current = d;
    return 0;
}
int hipDeviceGetAttribute(int* v, int, int) {
    *v = 256;
    return 0;
}
int hipDeviceSynchronize() { return 0; }
int hipGetLastError() {
    const int e = last_error;
    last_error = 0;
    return e;
}
const char* hipGetErrorString(int) { return "fake error"; }
int hipMemGetInfo(size_t* f, size_t* t) {
    *f = free_bytes;
    *t = (size_t)1 << 39;
    return 0;
}

// ---- memory ----
int hipMalloc(void** p, size_t n) {
    *p = nullptr;
    if (fails("hipMalloc")) return err(2);
    *p = std::calloc(n ? n : 1, 1);
    count("malloc");
    count(on_device("malloc"));
    count(on_device("bytes"), (long long)n);
    count("bytes", (long long)n);
    std::lock_guard<std::mutex> g(lock);
    sizes[*p] = n;
    return 0;
}
int hipFree(void* p) {
    std::lock_guard<std::mutex> g(lock);
    auto it = sizes.find(p);
    if (it == sizes.end()) {
        counters["bad free"] += p != nullptr;
        return 0;
    }
    counters["bytes"] -= (long long)it->second;
    sizes.erase(it);
    std::free(p);
    return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned) {
    *p = nullptr;
    if (fails("hipHostMalloc")) return err(2);
    *p = std::calloc(n ? n : 1, 1);
    count("pinned bytes", (long long)n);
    std::lock_guard<std::mutex> g(lock);
    sizes[*p] = n;
    return 0;
}
int hipHostFree(void* p) {
    std::lock_guard<std::mutex> g(lock);
    auto it = sizes.find(p);
    if (it != sizes.end()) {
        counters["pinned bytes"] -= (long long)it->second;
        sizes.erase(it);
        std::free(p);
    }
    return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int) {
    std::memcpy(d, s, n);
    return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) {
    std::memcpy(d, s, n);
    return 0;
}
int hipMemset(void* d, int v, size_t n) {
    std::memset(d, v, n);
    return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void*) {
    std::memset(d, v, n);
    return 0;
}
int hipGetSymbolAddress(void**, const void*) { return err(1); }

// ---- streams, events, graphs ----
int hipStreamCreateWithFlags(void** s, unsigned) {
    *s = new Object{current};
    return 0;
}
int hipStreamDestroy(void* s) {
    delete static_cast<Object*>(s);
    return 0;
}
int hipStreamSynchronize(void*) {
    count("stream sync");
    return 0;
}
int hipEventCreate(void** e) {
    *e = new Object{current};
    count("event");
    return 0;
}
int hipEventCreateWithFlags(void** e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void* e) {
    delete static_cast<Object*>(e);
    return 0;
}
int hipEventRecord(void* e, void* s) {
    if (s && static_cast<Object*>(e)->device != static_cast<Object*>(s)->device) {
        ++wrong_device;
        return err(400);
    }
    return 0;
}
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*) {
    *ms = 1.0f;
    return 0;
}
int hipThreadExchangeStreamCaptureMode(int*) { return 0; }
thread_local bool capturing = false;
int hipStreamBeginCapture(void*, int) {
    count("capture");
    capturing = true;
    return 0;
}
int hipStreamEndCapture(void*, void** g) {
    capturing = false;
    *g = new Object{current};
    return 0;
}
int hipGraphInstantiate(void** x, void*, void*, char*, size_t) {
    *x = new Object{current};
    return 0;
}
int hipGraphLaunch(void*, void*) {
    count("replay");
    return 0;
}
int hipGraphDestroy(void* g) {
    delete static_cast<Object*>(g);
    return 0;
}
int hipGraphExecDestroy(void* x) {
    delete static_cast<Object*>(x);
    return 0;
}

// ---- kernels ----
struct Dim3 {
    uint32_t x, y, z;
};
thread_local struct {
    Dim3 grid, block;
    size_t shared;
    void* stream;
} call;

void** __hipRegisterFatBinary(const void*) {
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    kernels[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
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
int hipLaunchKernel(const void* f, Dim3, Dim3, void** args, size_t, void*) {
    // k_name in the mangled name, up to its template arguments or its end
    const std::string& m = kernels[f];
    const size_t at = m.find("k_");
    const std::string name = at == std::string::npos ? m : m.substr(at, m.find_first_of("IE", at) - at);
    count("kernel " + name);
    count("mangled " + m);
    count(capturing ? "captured" : "kernels");
    if (name == "k_read_xyz") {
        const uint32_t n = *static_cast<uint32_t*>(args[0]);
        const float* src = *static_cast<float**>(args[1]);
        const uint32_t* oid = *static_cast<uint32_t**>(args[2]);
        float* out = *static_cast<float**>(args[3]);
        for (uint32_t i = 0; i < n; ++i)
            for (int a = 0; a < 3; ++a) out[3 * (size_t)oid[i] + a] = src[4 * (size_t)i + a];
    }
    return 0;
}

}  // extern "C"
