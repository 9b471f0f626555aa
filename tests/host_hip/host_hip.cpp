// A model of the HIP runtime in host memory, for tests of the library's host
// code (allocation, error and ordering paths) where there is no GPU. It stands
// in for libamdhip64 (same soname), so a process that loads it first runs
// libchimera_hip.so on it. "Device" memory is lazily mapped host memory of a
// set capacity; kernels do nothing but be counted, except those in run();
// work on a stream waits until something waits for it, while calls on the
// null stream run at once (the library's streams are non-blocking ones). The
// last error stays set until hipGetLastError reads it.
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>

#include <cstdint>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

namespace {

std::recursive_mutex g_mu;
using Lock = std::lock_guard<std::recursive_mutex>;

struct Stream {
    std::deque<std::function<void()>> queue;
};
struct Event {
    Stream* stream = nullptr;
    uint64_t recorded = 0, reached = 0;
};

std::vector<Stream*> g_streams;
std::map<void*, size_t> g_blocks;
size_t g_capacity = size_t{1} << 34, g_used = 0, g_peak = 0;
size_t g_refuse_from = 0, g_refuse_to = 0;  // hipMalloc sizes that fail (to > 0)
int g_refuse_host = 0, g_refuse_pointer = 0, g_cus = 256;
thread_local hipError_t g_last = hipSuccess;
std::map<const void*, std::string> g_names;
std::map<const void*, std::pair<size_t, void*>> g_vars;
std::map<std::string, int> g_launches;
std::map<std::string, int> g_threads;  // of the last launch of each kernel
int g_lane_cap = -1;
std::vector<size_t> g_sizes;  // of every successful hipMalloc, in order

struct Config {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
};
thread_local std::vector<Config> g_config;

hipError_t done(hipError_t e) {
    if (e != hipSuccess) g_last = e;
    return e;
}

void* map_bytes(size_t n) {
    void* p = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    return p == MAP_FAILED ? nullptr : p;
}

void drain(Stream* s) {
    while (!s->queue.empty()) {
        auto f = std::move(s->queue.front());
        s->queue.pop_front();
        f();
    }
}

void push(hipStream_t s, std::function<void()> f) {
    if (s == nullptr)
        f();
    else
        reinterpret_cast<Stream*>(s)->queue.push_back(std::move(f));
}

size_t rounded(size_t n) { return (n + 4095) / 4096 * 4096; }

// The kernels whose effect a test needs.
std::function<void()> run(const std::string& name, void** args) {
    if (name.find("invert_kernel") != std::string::npos) {  // (inv, n, pos)
        const auto* inv = *static_cast<const uint32_t**>(args[0]);
        const int64_t n = *static_cast<int64_t*>(args[1]);
        auto* pos = *static_cast<uint32_t**>(args[2]);
        return [=] {
            for (int64_t p = 0; p < n; ++p) pos[inv[p]] = static_cast<uint32_t>(p);
        };
    }
    if (name.find("cluster_bounds_kernel") != std::string::npos) {  // (sorted, n, k, cluster_pos): clusters of one size
        const int64_t n = *static_cast<int64_t*>(args[1]), k = *static_cast<int64_t*>(args[2]);
        auto* pos = *static_cast<uint64_t**>(args[3]);
        return [=] {
            for (int64_t c = 0; c <= k; ++c) pos[c] = static_cast<uint64_t>(n * c / k);
        };
    }
    return [] {};
}

}  // namespace

extern "C" {

// ---- controls ----
void host_hip_set_capacity(size_t bytes) { g_capacity = bytes; }
void host_hip_set_cus(int n) { g_cus = n; }
void host_hip_refuse_malloc(size_t from, size_t to) { g_refuse_from = from, g_refuse_to = to; }
void host_hip_refuse_host(int n) { g_refuse_host = n; }        // the next n hipHostMalloc calls fail
void host_hip_refuse_pointer(int n) { g_refuse_pointer = n; }  // the next n hipHostGetDevicePointer calls fail
size_t host_hip_used(void) { return g_used; }
size_t host_hip_peak(void) { return g_peak; }
void host_hip_reset_peak(void) { g_peak = g_used; }
// bytes asked for by the hipMalloc call `back` calls before the last
size_t host_hip_malloc(int back) { return g_sizes[g_sizes.size() - 1 - static_cast<size_t>(back)]; }
// launches of kernels whose name holds `part`
int host_hip_launches(const char* part) {
    Lock lock(g_mu);
    int n = 0;
    for (const auto& l : g_launches)
        if (l.first.find(part) != std::string::npos) n += l.second;
    return n;
}
void host_hip_reset_launches(void) {
    Lock lock(g_mu);
    g_launches.clear();
    g_threads.clear();
}
// threads per block of the last launch of a kernel whose name holds `part` (0: none)
int host_hip_threads(const char* part) {
    Lock lock(g_mu);
    for (const auto& l : g_threads)
        if (l.first.find(part) != std::string::npos) return l.second;
    return 0;
}
// candidates per sub-list in the last launch of the assignment's rerank (its argument 6)
int host_hip_lane_cap(void) { return g_lane_cap; }

// ---- modules and launches ----
void** __hipRegisterFatBinary(const void*) {
    static void* module = nullptr;
    return &module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, dim3*, dim3*,
                           int*) {
    g_names[host] = name;
}
void __hipRegisterVar(void**, void* var, char*, char*, int, size_t size, int, int) { g_vars[var] = {size, nullptr}; }

hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
    g_config.push_back({grid, block, shared, stream});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream) {
    const Config c = g_config.back();
    g_config.pop_back();
    *grid = c.grid;
    *block = c.block;
    *shared = c.shared;
    *stream = c.stream;
    return hipSuccess;
}

hipError_t hipLaunchKernel(const void* function, dim3 grid, dim3 block, void** args, size_t, hipStream_t stream) {
    Lock lock(g_mu);
    if (grid.x == 0 || grid.y == 0 || grid.z == 0 || block.x * block.y * block.z == 0 ||
        block.x * block.y * block.z > 1024)
        return done(hipErrorInvalidConfiguration);
    const std::string& name = g_names[function];
    ++g_launches[name];
    g_threads[name] = static_cast<int>(block.x * block.y * block.z);
    if (name.find("probe_top1_rerank_kernel") != std::string::npos) g_lane_cap = *static_cast<int*>(args[6]);
    push(stream, run(name, args));
    return hipSuccess;
}

hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }

// ---- devices ----
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = g_cus, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->gcnArchName, "gfx950:sramecc+:xnack-");
    p->multiProcessorCount = g_cus;
    p->warpSize = 64;
    p->maxThreadsPerBlock = 1024;
    return hipSuccess;
}
int hipGetStreamDeviceId(hipStream_t) { return 0; }
const char* hipGetErrorString(hipError_t e) {
    return e == hipErrorOutOfMemory ? "out of memory" : e == hipSuccess ? "no error" : "error";
}
hipError_t hipGetLastError(void) {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}

// ---- memory ----
hipError_t hipMalloc(void** p, size_t n) {
    Lock lock(g_mu);
    *p = nullptr;
    const size_t bytes = rounded(n);
    if (g_used + bytes > g_capacity || (n >= g_refuse_from && n <= g_refuse_to && g_refuse_to > 0))
        return done(hipErrorOutOfMemory);
    *p = map_bytes(bytes);
    if (!*p) return done(hipErrorOutOfMemory);
    g_blocks[*p] = bytes;
    g_sizes.push_back(n);
    g_used += bytes;
    if (g_used > g_peak) g_peak = g_used;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    Lock lock(g_mu);
    for (Stream* s : g_streams) drain(s);
    if (!p) return hipSuccess;
    const auto it = g_blocks.find(p);
    if (it == g_blocks.end()) return done(hipErrorInvalidValue);
    munmap(p, it->second);
    g_used -= it->second;
    g_blocks.erase(it);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* free_bytes, size_t* total) {
    *free_bytes = g_capacity - g_used;
    *total = g_capacity;
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    Lock lock(g_mu);
    *p = nullptr;
    if (g_refuse_host > 0) {
        --g_refuse_host;
        return done(hipErrorOutOfMemory);
    }
    *p = map_bytes(rounded(n));
    g_blocks[*p] = rounded(n);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    Lock lock(g_mu);
    const auto it = g_blocks.find(p);
    if (it == g_blocks.end()) return done(hipErrorInvalidValue);
    munmap(p, it->second);
    g_blocks.erase(it);
    return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) {
    Lock lock(g_mu);
    if (g_refuse_pointer > 0) {
        --g_refuse_pointer;
        return done(hipErrorInvalidValue);
    }
    return *d = h, hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* symbol) {
    Lock lock(g_mu);
    auto& v = g_vars[symbol];
    if (!v.second) v.second = map_bytes(rounded(v.first));
    return *p = v.second, hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t stream) {
    Lock lock(g_mu);
    push(stream, [=] { std::memcpy(d, s, n); });
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind kind) {
    return hipMemcpyAsync(d, s, n, kind, nullptr);
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t stream) {
    Lock lock(g_mu);
    push(stream, [=] { std::memset(d, v, n); });
    return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) { return hipMemsetAsync(d, v, n, nullptr); }

// ---- streams, events, graphs ----
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    Lock lock(g_mu);
    g_streams.push_back(new Stream);
    *s = reinterpret_cast<hipStream_t>(g_streams.back());
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    Lock lock(g_mu);
    drain(reinterpret_cast<Stream*>(s));
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    Lock lock(g_mu);
    if (s) drain(reinterpret_cast<Stream*>(s));
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    return *e = reinterpret_cast<hipEvent_t>(new Event), hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    Lock lock(g_mu);
    auto* ev = reinterpret_cast<Event*>(e);
    ev->stream = reinterpret_cast<Stream*>(s);
    const uint64_t id = ++ev->recorded;
    push(s, [=] { ev->reached = id; });
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    Lock lock(g_mu);
    auto* ev = reinterpret_cast<Event*>(e);
    while (ev->reached < ev->recorded && !ev->stream->queue.empty()) {
        auto f = std::move(ev->stream->queue.front());
        ev->stream->queue.pop_front();
        f();
    }
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0.0f, hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return done(hipErrorNotSupported); }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return done(hipErrorNotSupported); }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    return done(hipErrorNotSupported);
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return done(hipErrorNotSupported); }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

}  // extern "C"
