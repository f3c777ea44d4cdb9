// A HIP runtime on the CPU for the tests of the library's host code: device
// memory is host memory (a new block's words hold 2654435761 times their
// index), kernels do nothing but rh_read_back, which copies when the test's
// gate opens, rh_reduce_counters, which counts nothing, and rh_box_classes.  Loaded with global symbols before the library,
// in a process of its own.  fake_* set it up and report what was called.
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <thread>

namespace {

struct Stream {
    int dev;
    std::mutex m;
    std::condition_variable idle;
    int pending = 0;
    bool failed = false;
};

struct Block {
    size_t bytes;
    int dev;                              // -1: pinned host memory
};

thread_local int t_dev = 0;
std::mutex g_m;
std::condition_variable g_gateCv;
int g_gate = -1;                          // workgroups of each copy let through (-1: all)
bool g_lose = false;
bool g_refusePinned = false, g_boxVaries = false;
std::map<void*, Block> g_blocks;
std::map<const void*, std::string> g_kernels;
size_t g_most = SIZE_MAX;                 // bytes of the largest allocation granted
std::atomic<uint32_t> g_noRoom{0};        // transparent hits the next frame has no room for
std::atomic<int> g_deviceSyncs{0}, g_pinnedCalls{0}, g_plainCopies{0}, g_waiting{0}, g_streamWaits{0}, g_pinnedCopies{0};

struct Config { dim3 grid, wg; size_t lds; hipStream_t st; };
thread_local Config t_config;

hipError_t take(void** p, size_t bytes, int dev) {
    if (bytes > g_most) return hipErrorOutOfMemory;
    // (of more than a gigabyte only the first words are there: nothing reads them)
    const size_t real = bytes > (size_t(1) << 30) ? 4096 : bytes;
    void* q = std::aligned_alloc(256, (real + 255) / 256 * 256);
    if (!q) return hipErrorOutOfMemory;
    for (size_t i = 0; i < real / 4; ++i) static_cast<uint32_t*>(q)[i] = (uint32_t)i * 2654435761u;
    std::lock_guard<std::mutex> lk(g_m);
    g_blocks[q] = Block{bytes, dev};
    *p = q;
    return hipSuccess;
}

hipError_t give(void* p) {
    if (!p) return hipSuccess;
    {
        std::lock_guard<std::mutex> lk(g_m);
        if (!g_blocks.erase(p)) return hipErrorInvalidValue;
    }
    std::free(p);
    return hipSuccess;
}

Stream* S(hipStream_t s) { return reinterpret_cast<Stream*>(s); }

// rh_read_back(src, dst, bytes, flags, seq), a workgroup at a time
void read_back(Stream* st, unsigned grid, const char* src, char* dst, size_t bytes, volatile uint32_t* flags, uint32_t seq) {
    const size_t per = 16384;
    for (unsigned w = 0; w < grid && !g_lose; ++w) {
        {
            std::unique_lock<std::mutex> lk(g_m);
            auto open = [w] { return g_gate < 0 || (int)w < g_gate; };
            if (!open()) {
                ++g_waiting;
                g_gateCv.wait(lk, open);
                --g_waiting;
            }
        }
        std::memcpy(dst + w * per, src + w * per, std::min(per, bytes - w * per));
        std::atomic_thread_fence(std::memory_order_release);
        flags[w] = seq;
    }
    std::lock_guard<std::mutex> lk(st->m);
    st->failed = g_lose;
    if (--st->pending == 0) st->idle.notify_all();
}

}  // namespace

extern "C" {

void fake_gate(int workgroups) {
    std::lock_guard<std::mutex> lk(g_m);
    g_gate = workgroups;
    g_gateCv.notify_all();
}
void fake_most(uint64_t bytes) { g_most = bytes; }
void fake_no_room(uint32_t n) { g_noRoom = n; }
void fake_lose(int on) { g_lose = on != 0; }
void fake_box_varies(int on) { g_boxVaries = on != 0; }
void fake_refuse_pinned(int on) { g_refusePinned = on != 0; }
int fake_waiting() { return g_waiting; }
int fake_device_syncs() { return g_deviceSyncs; }
int fake_pinned_calls() { return g_pinnedCalls; }
int fake_stream_waits() { return g_streamWaits; }
int fake_pinned_copies() { return g_pinnedCopies; }
int fake_plain_copies() { return g_plainCopies; }
// bytes held: of a device, or pinned (-1)
uint64_t fake_held(int dev) {
    std::lock_guard<std::mutex> lk(g_m);
    uint64_t n = 0;
    for (const auto& b : g_blocks) n += b.second.dev == dev ? b.second.bytes : 0;
    return n;
}

void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    g_kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 wg, size_t lds, hipStream_t st) {
    t_config = Config{grid, wg, lds, st};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* wg, size_t* lds, hipStream_t* st) {
    *grid = t_config.grid;
    *wg = t_config.wg;
    *lds = t_config.lds;
    *st = t_config.st;
    return hipSuccess;
}

hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void** args, size_t, hipStream_t st) {
    const std::string& name = g_kernels[f];
    if (name.find("rh_reduce_counters") != std::string::npos) {
        // no hits but those without room: rh_reduce_counters(rows, nrows, refs,
        // nbuckets, counters, hitCtl, host)
        std::memset(*static_cast<void**>(args[4]), 0, 9 * 8);
        uint32_t* ctl = *static_cast<uint32_t**>(args[5]);
        std::memset(ctl, 0, 4 * 4);
        ctl[0] = g_noRoom.exchange(0);
        if (unsigned long long* host = *static_cast<unsigned long long**>(args[6])) {
            std::memset(host, 0, 13 * 8);
            host[9] = ctl[0];
        }
    }
    if (name.find("rh_box_classes") != std::string::npos) {
        // rh_box_classes(frame, patterns, positions, rows): every test may hold, and does not always or does
        uint32_t* rows = *static_cast<uint32_t**>(args[3]);
        for (unsigned i = 0; i < grid.x * 64; ++i) rows[i] = g_boxVaries ? 0xffff0000u : 0xffffffffu;
    }
    if (name.find("rh_read_back") == std::string::npos) return hipSuccess;
    Stream* s = S(st);
    {
        std::lock_guard<std::mutex> lk(s->m);
        ++s->pending;
    }
    std::thread(read_back, s, grid.x, *static_cast<const char**>(args[0]), *static_cast<char**>(args[1]),
                *static_cast<size_t*>(args[2]), *static_cast<volatile uint32_t**>(args[3]),
                *static_cast<uint32_t*>(args[4]))
        .detach();
    return hipSuccess;
}

hipError_t hipGetDeviceCount(int* n) { *n = 2; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = t_dev; return hipSuccess; }
hipError_t hipSetDevice(int d) { t_dev = d; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipDeviceSynchronize() { ++g_deviceSyncs; return hipSuccess; }
hipError_t hipDeviceGetDefaultMemPool(hipMemPool_t* p, int) { *p = nullptr; return hipSuccess; }
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void*) { return hipSuccess; }
hipError_t hipMemPoolTrimTo(hipMemPool_t, size_t) { return hipSuccess; }

hipError_t hipMalloc(void** p, size_t n) { return take(p, n, t_dev); }
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t st) { return take(p, n, S(st)->dev); }
hipError_t hipFree(void* p) { return give(p); }
hipError_t hipFreeAsync(void* p, hipStream_t) { return give(p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    ++g_pinnedCalls;
    return g_refusePinned ? hipErrorOutOfMemory : take(p, n, -1);
}
hipError_t hipHostFree(void* p) { return give(p); }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static unsigned char scratch[4 << 20];
    *p = scratch;
    return hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n) { std::memset(p, v, n); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) {
    if (k == hipMemcpyDeviceToHost) {
        ++g_plainCopies;
        std::lock_guard<std::mutex> lk(g_m);
        auto b = g_blocks.upper_bound(d);
        if (b != g_blocks.begin() && (--b)->second.dev < 0 && static_cast<char*>(b->first) + b->second.bytes > d) ++g_pinnedCopies;
    }
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    Stream* n = new Stream();
    n->dev = t_dev;
    *s = reinterpret_cast<hipStream_t>(n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    ++g_streamWaits;
    std::unique_lock<std::mutex> lk(S(s)->m);
    S(s)->idle.wait(lk, [&] { return S(s)->pending == 0; });
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t s) {
    std::lock_guard<std::mutex> lk(S(s)->m);
    return S(s)->pending ? hipErrorNotReady : (S(s)->failed ? hipErrorUnknown : hipSuccess);
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) { return hipErrorNotSupported; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = reinterpret_cast<hipEvent_t>(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* t, hipEvent_t, hipEvent_t) { *t = 0.0f; return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 2; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }

}  // extern "C"
