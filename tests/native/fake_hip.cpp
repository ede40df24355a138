// A HIP runtime on the host that runs no kernels, for tests of the library's
// host code: device memory is host memory, and every kernel launch is recorded
// with its thread, stream and grid.  Loaded with RTLD_GLOBAL before
// libleafhip.so, whose HIP calls then bind to it.
#include <atomic>
#include <chrono>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <thread>

struct dim3 { uint32_t x, y, z; };
typedef void* stream_t;
enum { kSuccess = 0, kOutOfMemory = 2, kCaptureImplicit = 906 };

static std::mutex g_lock;
static std::string g_log;
static std::map<const void*, std::string>& names() {
    static auto* m = new std::map<const void*, std::string>();   // kernels register before main
    return *m;
}
static std::atomic<int> g_capturing{0}, g_delay_us{0};
static std::atomic<size_t> g_malloc_limit{SIZE_MAX};
static thread_local int t_error = kSuccess;
struct Config { dim3 grid, block; size_t shared; stream_t stream; };
static thread_local Config t_config;

static void record(const char* what, const std::string& rest) {
    const auto thread = std::hash<std::thread::id>()(std::this_thread::get_id());
    std::lock_guard<std::mutex> guard(g_lock);
    g_log += std::string(what) + " " + std::to_string(thread) + " " + rest + "\n";
}

extern "C" {
// ---- the tests' side
void fake_reset() { std::lock_guard<std::mutex> guard(g_lock); g_log.clear(); }
size_t fake_log(char* out, size_t capacity) {
    std::lock_guard<std::mutex> guard(g_lock);
    const size_t n = g_log.size() < capacity ? g_log.size() : capacity;
    std::memcpy(out, g_log.data(), n);
    return g_log.size();
}
void fake_set_capturing(int on) { g_capturing = on; }
void fake_set_launch_delay_us(int us) { g_delay_us = us; }
void fake_set_malloc_limit(size_t bytes) { g_malloc_limit = bytes; }   // larger allocations fail

// ---- HIP's
void** __hipRegisterFatBinary(const void*) { static void* handle; return &handle; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    names()[host] = name;
}
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, stream_t stream) {
    t_config = Config{grid, block, shared, stream};
    return kSuccess;
}
int __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, stream_t* stream) {
    *grid = t_config.grid; *block = t_config.block; *shared = t_config.shared; *stream = t_config.stream;
    return kSuccess;
}
int hipLaunchKernel(const void* f, dim3 grid, dim3, void**, size_t, stream_t stream) {
    char text[96];
    std::snprintf(text, sizeof text, " %p %u %u %u", stream, grid.x, grid.y, grid.z);
    record("launch", names()[f] + text);
    if (g_delay_us) std::this_thread::sleep_for(std::chrono::microseconds(g_delay_us));
    return kSuccess;
}
int hipLaunchCooperativeKernel(const void* f, dim3 grid, dim3 block, void** args, unsigned shared, stream_t stream) {
    return hipLaunchKernel(f, grid, block, args, shared, stream);
}
int hipMalloc(void** out, size_t bytes) {
    if (bytes > g_malloc_limit) return t_error = kOutOfMemory;
    *out = std::aligned_alloc(256, (bytes + 255) / 256 * 256);
    std::memset(*out, 0, bytes);
    return kSuccess;
}
int hipExtMallocWithFlags(void** out, size_t bytes, unsigned) { return hipMalloc(out, bytes); }
int hipHostMalloc(void** out, size_t bytes, unsigned) { return hipMalloc(out, bytes); }
int hipFree(void* p) { std::free(p); return kSuccess; }
int hipHostFree(void* p) { std::free(p); return kSuccess; }
int hipHostGetDevicePointer(void** out, void* p, unsigned) { *out = p; return kSuccess; }
int hipGetSymbolAddress(void** out, const void*) { static char array[1 << 10]; *out = array; return kSuccess; }
int hipMemcpy(void* dst, const void* src, size_t bytes, int) { std::memcpy(dst, src, bytes); return kSuccess; }
int hipMemcpyAsync(void* dst, const void* src, size_t bytes, int, stream_t) {
    record("copy", std::to_string(bytes));
    std::memcpy(dst, src, bytes);
    if (g_delay_us) std::this_thread::sleep_for(std::chrono::microseconds(g_delay_us));
    return kSuccess;
}
int hipMemcpy2DAsync(void* dst, size_t dpitch, const void* src, size_t spitch, size_t width, size_t height, int, stream_t) {
    for (size_t y = 0; y < height; ++y) std::memcpy((char*)dst + y * dpitch, (const char*)src + y * spitch, width);
    return kSuccess;
}
int hipMemset(void* p, int value, size_t bytes) { std::memset(p, value, bytes); return kSuccess; }
int hipMemsetAsync(void* p, int value, size_t bytes, stream_t) { return hipMemset(p, value, bytes); }
int hipStreamIsCapturing(stream_t stream, int* status) {
    if (!stream && g_capturing) return t_error = kCaptureImplicit;   // the null stream, beside a capture
    *status = g_capturing ? 1 : 0;
    return kSuccess;
}
int hipGetLastError() { const int e = t_error; t_error = kSuccess; return e; }
const char* hipGetErrorString(int) { return "fake HIP error"; }
int hipGetDevice(int* d) { *d = 0; return kSuccess; }
int hipSetDevice(int) { return kSuccess; }
int hipGetDeviceCount(int* n) { *n = 1; return kSuccess; }
int hipDeviceGetAttribute(int* v, int, int) { *v = 256; return kSuccess; }
int hipDeviceSynchronize() { return kSuccess; }
int hipFuncSetAttribute(const void*, int, int) { return kSuccess; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 1; return kSuccess; }
int hipStreamCreateWithFlags(stream_t* s, unsigned) { *s = std::malloc(1); return kSuccess; }
int hipStreamDestroy(stream_t s) { std::free(s); return kSuccess; }
int hipStreamSynchronize(stream_t) { return kSuccess; }
int hipStreamBeginCapture(stream_t, int) { return kSuccess; }
int hipStreamEndCapture(stream_t, void** g) { *g = nullptr; return kSuccess; }
int hipGraphInstantiate(void** e, void*, void*, char*, size_t) { *e = nullptr; return kSuccess; }
int hipGraphDestroy(void*) { return kSuccess; }
int hipGraphExecDestroy(void*) { return kSuccess; }
int hipGraphLaunch(void*, stream_t) { return kSuccess; }
int hipEventCreate(void** e) { *e = nullptr; return kSuccess; }
int hipEventDestroy(void*) { return kSuccess; }
int hipEventRecord(void*, stream_t) { return kSuccess; }
int hipEventSynchronize(void*) { return kSuccess; }
int hipEventElapsedTime(float* ms, void*, void*) { *ms = 0; return kSuccess; }
}
