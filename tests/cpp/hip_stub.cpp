// A double of the HIP runtime functions libhbem.so calls, for tests of the library's
// host code on machines without a GPU: device memory is host memory of a set
// capacity (reserved, not resident until written), copies are copies, kernels only
// enter a log, streams and events do nothing.  Loaded with RTLD_GLOBAL before
// libhbem.so, its definitions take precedence over the runtime's.
#include <sys/mman.h>

#include <cstdint>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

namespace {
struct Dim3 {
    uint32_t x, y, z;
};
constexpr int kOk = 0, kOutOfMemory = 2;
std::mutex mu;
std::map<void*, size_t> blocks;
std::map<const void*, std::string> names;
size_t capacity = (size_t)288 << 30, used = 0, peak = 0;
long fail_in = 0;               // > 0: that allocation from now on fails
std::string launches;
Dim3 grid, block;
size_t shared;
void* stream;

void* reserve(size_t n) {
    void* p = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    return p == MAP_FAILED ? nullptr : p;
}
}  // namespace

extern "C" {

// Test interface
void hip_stub_capacity(size_t bytes) { capacity = bytes; }
void hip_stub_fail(long n) { fail_in = n; }
long hip_stub_failing() { return fail_in; }
size_t hip_stub_used() { return used; }
size_t hip_stub_peak() {
    const size_t p = peak;
    peak = used;
    return p;
}
// the launches since the last call, one "kernel x y z" a line
const char* hip_stub_launches() {
    static std::string out;
    out.swap(launches);
    launches.clear();
    return out.c_str();
}

// Runtime interface
int hipMalloc(void** p, size_t n) {
    std::lock_guard<std::mutex> lk(mu);
    *p = nullptr;
    if (fail_in > 0 && --fail_in == 0) return kOutOfMemory;
    if (n == 0) return kOk;
    if (n > capacity - used) return kOutOfMemory;
    if (!(*p = reserve(n))) return kOutOfMemory;
    blocks[*p] = n;
    used += n;
    if (used > peak) peak = used;
    return kOk;
}
int hipFree(void* p) {
    std::lock_guard<std::mutex> lk(mu);
    auto it = blocks.find(p);
    if (it == blocks.end()) return p ? 1 : kOk;
    munmap(p, it->second);
    used -= it->second;
    blocks.erase(it);
    return kOk;
}
int hipMemGetInfo(size_t* fr, size_t* tot) {
    *fr = capacity - used;
    *tot = capacity;
    return kOk;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void*) {
    if (kind != 3) std::memcpy(d, s, n);          // device to device: nothing was computed there
    return kOk;
}
int hipMemsetAsync(void* d, int v, size_t n, void*) {
    std::memset(d, v, n);
    return kOk;
}
int hipLaunchKernel(const void* f, Dim3 g, Dim3, void**, size_t, void*) {
    std::lock_guard<std::mutex> lk(mu);
    launches += names[f] + " " + std::to_string(g.x) + " " + std::to_string(g.y) + " " + std::to_string(g.z) + "\n";
    return kOk;
}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t sh, void* st) {
    grid = g;
    block = b;
    shared = sh;
    stream = st;
    return kOk;
}
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* sh, void** st) {
    *g = grid;
    *b = block;
    *sh = shared;
    *st = stream;
    return kOk;
}
void** __hipRegisterFatBinary(const void*) {
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    names[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int hipGetSymbolAddress(void** p, const void*) {
    static void* mem = reserve((size_t)1 << 30);
    *p = mem;
    return kOk;
}
int hipGetDevice(int* d) {
    *d = 0;
    return kOk;
}
int hipGetDeviceCount(int* n) {
    *n = 1;
    return kOk;
}
int hipSetDevice(int) { return kOk; }
int hipGetLastError() { return kOk; }
const char* hipGetErrorString(int) { return "error"; }
int hipStreamCreateWithFlags(void** s, unsigned) {
    *s = (void*)1;
    return kOk;
}
int hipStreamDestroy(void*) { return kOk; }
int hipStreamSynchronize(void*) { return kOk; }
int hipStreamBeginCapture(void*, int) { return kOk; }
int hipStreamEndCapture(void*, void** g) {
    *g = (void*)1;
    return kOk;
}
int hipGraphInstantiate(void** e, void*, void*, char*, size_t) {
    *e = (void*)1;
    return kOk;
}
int hipGraphDestroy(void*) { return kOk; }
int hipGraphExecDestroy(void*) { return kOk; }
int hipGraphLaunch(void*, void*) { return kOk; }
int hipEventCreate(void** e) {
    *e = (void*)1;
    return kOk;
}
int hipEventDestroy(void*) { return kOk; }
int hipEventRecord(void*, void*) { return kOk; }
int hipEventSynchronize(void*) { return kOk; }
int hipEventElapsedTime(float* ms, void*, void*) {
    *ms = 0.f;
    return kOk;
}

}  // extern "C"
