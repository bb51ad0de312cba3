// A HIP runtime for tests of the host code without a GPU: allocations come from
// the host (zeroed), launches do nothing, and calls are recorded. Loaded with
// RTLD_GLOBAL before libgat.so, so that its symbols are taken for the real ones.
#include <hip/hip_runtime_api.h>

#include <chrono>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <thread>

namespace {
std::mutex mu;
std::condition_variable cv;
std::string log_text;
std::map<void *, size_t> live;
std::map<const void *, std::string> kernels;
size_t live_bytes = 0, limit = SIZE_MAX, refuse_from = SIZE_MAX;
int refusals = 0;  // the next allocations of at least refuse_from bytes to refuse (-1: all)
int hold = 0, held = 0, copy_ms = 0;
hipError_t last = hipSuccess;
struct Config {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
};
thread_local Config config;

void say(const std::string &s) { log_text += s + "\n"; }
}  // namespace

extern "C" {
// ---- what a test sets and reads
const char *fake_log() {  // everything recorded since the last call
    static thread_local std::string out;
    std::lock_guard<std::mutex> lk(mu);
    out.swap(log_text);
    log_text.clear();
    return out.c_str();
}
void fake_limit(size_t bytes) { limit = bytes; }  // of all live device memory
void fake_refuse(size_t from_bytes, int times) {
    refuse_from = from_bytes;
    refusals = times;
}
size_t fake_live() {
    std::lock_guard<std::mutex> lk(mu);
    return live_bytes;
}
void fake_slow_copies(int ms) { copy_ms = ms; }  // every copy takes so long
// While held, the first stream to be waited for does not finish.
void fake_hold() { hold = 1; }
int fake_held() {
    std::lock_guard<std::mutex> lk(mu);
    return held;
}
void fake_release() {
    std::lock_guard<std::mutex> lk(mu);
    hold = held = 0;
    cv.notify_all();
}

// ---- the runtime
hipError_t hipGetDeviceCount(int *n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    std::memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    p->sharedMemPerBlock = p->maxSharedMemoryPerMultiProcessor = 160 << 10;
    std::strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
    *v = 100000;
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t bytes) {
    std::lock_guard<std::mutex> lk(mu);
    *p = nullptr;
    const bool refused = bytes >= refuse_from && refusals != 0;
    if (refused && refusals > 0) refusals--;
    if (refused || live_bytes + bytes > limit) {
        say("refuse " + std::to_string(bytes));
        return last = hipErrorOutOfMemory;
    }
    *p = std::calloc(1, bytes ? bytes : 1);
    live[*p] = bytes;
    live_bytes += bytes;
    say("malloc " + std::to_string(bytes));
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    std::lock_guard<std::mutex> lk(mu);
    const auto it = live.find(p);
    if (it == live.end()) return p ? hipErrorInvalidValue : hipSuccess;
    live_bytes -= it->second;
    say("free " + std::to_string(it->second));
    live.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) {
    *p = std::calloc(1, bytes);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    if (copy_ms) std::this_thread::sleep_for(std::chrono::milliseconds(copy_ms));
    std::memcpy(d, s, n);
    std::lock_guard<std::mutex> lk(mu);
    say("copy " + std::to_string(n));
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    std::free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    std::unique_lock<std::mutex> lk(mu);
    if (hold && !held) {
        held = 1;
        cv.wait(lk, [] { return !hold; });
    }
    say("synchronized");
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) {
    *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    std::free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    std::lock_guard<std::mutex> lk(mu);
    say("event " + std::to_string(reinterpret_cast<size_t>(e)));
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) {
    std::lock_guard<std::mutex> lk(mu);
    say("elapsed " + std::to_string(reinterpret_cast<size_t>(a)) + " " + std::to_string(reinterpret_cast<size_t>(b)));
    *ms = 1.f;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
    *g = reinterpret_cast<hipGraph_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t) {
    *x = reinterpret_cast<hipGraphExec_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) {
    std::free(g);
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t g) {
    std::free(g);
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
    *p = nullptr;
    return hipErrorInvalidSymbol;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **, size_t, hipStream_t) {
    std::lock_guard<std::mutex> lk(mu);
    if (!grid.x || !block.x) return last = hipErrorInvalidConfiguration;
    say("launch " + kernels[f]);
    return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
    config = {grid, block, lds, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *s) {
    *grid = config.grid;
    *block = config.block;
    *lds = config.lds;
    *s = config.stream;
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) {
    static void *module;
    return &module;
}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *,
                           int *) {
    std::lock_guard<std::mutex> lk(mu);
    kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void **) {}
}  // extern "C"
