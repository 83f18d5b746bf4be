// A host-only stand-in for the HIP runtime and the rocBLAS calls of
// libvbm3d_hip.so, for tests of its host logic where memory is short or a
// launch fails.  Loaded with RTLD_GLOBAL before the library, its symbols are
// the ones the library binds.  Kernels and copies do nothing; allocations come
// out of `capacity` bytes; every call of interest is counted or logged.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <vector>

namespace {
size_t capacity = (size_t)1 << 40, used = 0, peak = 0;
std::map<void*, size_t> blocks;
int last_error = 0;
long launches = 0, fail_launch = -1;
// host buffers with a copy in flight: copies since the stream they are on was waited for
std::map<void*, long> in_flight;
long h2d = 0;
struct Cfg {
    uint32_t g[3], b[3];
    size_t shmem;
    void* stream;
};
std::vector<Cfg> pushed;
int err(int e) {
    if (e) last_error = e;
    return e;
}
}  // namespace

extern "C" {
void fake_reset(size_t cap, long fail_at) {
    capacity = cap;
    peak = used;
    launches = 0;
    fail_launch = fail_at;
    h2d = 0;
    last_error = 0;
}
size_t fake_used() { return used; }
size_t fake_peak() { return peak; }
long fake_launches() { return launches; }
long fake_h2d() { return h2d; }
long fake_in_flight() {
    long n = 0;
    for (auto& q : in_flight) n += q.second;
    return n;
}

void** __hipRegisterFatBinary(const void*) {
    static void* m;
    return &m;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
struct D3 {
    uint32_t x, y, z;
};
int __hipPushCallConfiguration(D3 g, D3 b, size_t sh, void* s) {
    pushed.push_back(Cfg{{g.x, g.y, g.z}, {b.x, b.y, b.z}, sh, s});
    return 0;
}
int __hipPopCallConfiguration(D3* g, D3* b, size_t* sh, void** s) {
    const Cfg c = pushed.back();
    pushed.pop_back();
    *g = D3{c.g[0], c.g[1], c.g[2]};
    *b = D3{c.b[0], c.b[1], c.b[2]};
    *sh = c.shmem;
    *s = c.stream;
    return 0;
}
int hipLaunchKernel(const void*, D3, D3, void**, size_t, void*) { return err(launches++ == fail_launch ? 719 : 0); }
int hipGetLastError() {
    const int e = last_error;
    last_error = 0;
    return e;
}
const char* hipGetErrorString(int) { return "fake error"; }
int hipMalloc(void** p, size_t n) {
    *p = nullptr;
    if (used + n > capacity) return err(2);
    void* q = std::malloc(n ? n : 1);  // untouched pages cost nothing
    if (!q) return err(2);
    blocks[q] = n;
    used += n;
    if (used > peak) peak = used;
    *p = q;
    return 0;
}
int hipFree(void* p) {
    in_flight.clear();  // waits for the device
    auto it = blocks.find(p);
    if (it == blocks.end()) return p ? err(1) : 0;
    used -= it->second;
    blocks.erase(it);
    std::free(p);
    return 0;
}
int hipMemGetInfo(size_t* fr, size_t* tot) {
    *fr = capacity - used;
    *tot = capacity;
    return 0;
}
int hipMemcpyAsync(void*, const void*, size_t, int kind, void* s) {
    if (kind == 1) h2d++;
    if (kind == 1 || kind == 2) in_flight[s]++;
    return 0;
}
int hipMemcpy(void*, const void*, size_t, int) { return 0; }
int hipMemset(void*, int, size_t) { return 0; }
int hipMemsetAsync(void*, int, size_t, void*) { return 0; }
int hipStreamSynchronize(void* s) {
    in_flight.erase(s);
    return 0;
}
int hipDeviceSynchronize() {
    in_flight.clear();
    return 0;
}
int hipStreamCreate(void** s) {
    *s = std::malloc(1);
    return 0;
}
int hipStreamDestroy(void* s) {
    std::free(s);
    return 0;
}
int hipStreamWaitEvent(void*, void*, unsigned) { return 0; }
int hipEventCreate(void** e) {
    *e = std::malloc(1);
    return 0;
}
int hipEventCreateWithFlags(void** e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void* e) {
    std::free(e);
    return 0;
}
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*) {
    *ms = 1.f;
    return 0;
}
int hipSetDevice(int) { return 0; }
int hipGetDevice(int* d) {
    *d = 0;
    return 0;
}
int hipDeviceGetAttribute(int* v, int, int) {
    *v = 256;
    return 0;
}
int hipGetSymbolAddress(void** p, const void*) {
    static void* a = std::malloc((size_t)256 << 20);
    *p = a;
    return 0;
}
int hipStreamBeginCapture(void*, int) { return 0; }
int hipStreamEndCapture(void*, void** g) {
    *g = nullptr;
    return 0;
}
int hipGraphInstantiate(void** x, void*, void*, char*, size_t) {
    *x = nullptr;
    return 0;
}
int hipGraphLaunch(void*, void*) { return 0; }
int hipGraphDestroy(void*) { return 0; }
int hipGraphExecDestroy(void*) { return 0; }
int rocblas_create_handle(void** h) {
    *h = std::malloc(1);
    return 0;
}
int rocblas_destroy_handle(void* h) {
    std::free(h);
    return 0;
}
int rocblas_set_stream(void*, void*) { return 0; }
int rocblas_dgemm_strided_batched(...) { return 0; }
const char* rocblas_status_to_string(int) { return "fake"; }
}
