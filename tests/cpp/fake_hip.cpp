// A stand-in for the HIP runtime entry points that libmiq.so calls, for tests
// of its host side without a GPU: kernels are not run but recorded (name, grid,
// the library buffers that their argument block points to), allocations are
// addresses that nothing reads, and the test sets the device's size, whether a
// stream captures, and the largest allocation that succeeds.  Loaded with
// RTLD_GLOBAL ahead of libmiq.so, its symbols take the runtime's place.
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
struct Launch {
    std::string name;
    dim3 grid, block;
    void *stream;
    std::vector<uint64_t> args;  // first 128 bytes of the first argument (an argument block or a scalar)
};
std::map<const void *, std::string> g_names;
std::vector<Launch> g_launches;
std::map<uint64_t, uint64_t> g_allocs;  // address -> bytes
uint64_t g_next = 0x7A0000000000ull;
size_t g_limit = SIZE_MAX;
bool g_capturing = false;
hipError_t g_last = hipSuccess;  // as the runtime's: an error stays until it is read
struct Config {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
} g_cfg;
}  // namespace

extern "C" {
// ---- the test's side
void fake_reset() { g_launches.clear(); }
void fake_capturing(int on) { g_capturing = on; }
void fake_malloc_limit(size_t bytes) { g_limit = bytes; }
int fake_launches() { return (int)g_launches.size(); }
const char *fake_name(int i) { return g_launches[i].name.c_str(); }
unsigned fake_blocks(int i) { return g_launches[i].grid.x * g_launches[i].grid.y * g_launches[i].grid.z; }
// k-th library buffer in launch i's arguments (0: no more)
uint64_t fake_buffer(int i, int k) {
    for (uint64_t v : g_launches[i].args) {
        auto it = g_allocs.upper_bound(v);
        if (it == g_allocs.begin()) continue;
        --it;
        if (v < it->first + it->second && k-- == 0) return it->first;
    }
    return 0;
}
uint64_t fake_allocated() {
    uint64_t n = 0;
    for (auto &a : g_allocs) n += a.second;
    return n;
}

// ---- the runtime's side
void **__hipRegisterFatBinary(const void *) {
    static void *h;
    return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *fn, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *, int *) {
    g_names[fn] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream) {
    g_cfg = Config{grid, block, lds, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *stream) {
    *grid = g_cfg.grid;
    *block = g_cfg.block;
    *lds = g_cfg.lds;
    *stream = g_cfg.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *fn, dim3 grid, dim3 block, void **args, size_t, hipStream_t stream) {
    Launch l{g_names[fn], grid, block, (void *)stream, std::vector<uint64_t>(16)};
    memcpy(l.args.data(), args[0], 128);
    g_launches.push_back(l);
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t bytes) {
    if (bytes > g_limit) return g_last = hipErrorOutOfMemory;
    *p = (void *)g_next;
    g_allocs[g_next] = bytes;
    g_next += (bytes + 0xFFFFFF) & ~(size_t)0xFFFFF;
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t) { return "fake HIP error"; }
hipError_t hipGetDevice(int *d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
    *v = 256;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) {
    *s = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
    *p = (void *)0x790000000000ull;
    return hipSuccess;
}
}
