// host_hip.cpp -- a stand-in for the HIP runtime, so that what libvz.so does on
// the host (what it allocates and when, the order of its calls, its locking)
// can be tested without a GPU.  Loaded globally before libvz.so, its symbols
// come before libamdhip64.so's.  Device memory is host memory (zeroed, with an
// optional limit), copies are done at once, kernels are noted and not run.
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>

#include <algorithm>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>
#include <string>

namespace {

struct Ev {
    bool timed, done = true;
};

std::mutex mu;
std::map<void*, size_t> blocks;
size_t used = 0, peak = 0, limit = ~(size_t)0;
std::map<const void*, std::string> kernels;
std::string log_text;
std::map<std::string, unsigned> launches;
bool hold = false;
std::deque<Ev*> held;
void (*on_free)() = nullptr;
size_t on_free_bytes = ~(size_t)0;

void note(const std::string& s) { log_text += s + "\n"; }

hipError_t alloc(void** p, size_t n, bool device)
{
    std::lock_guard<std::mutex> lk(mu);
    if (device && used + n > limit) {
        note("refuse " + std::to_string(n));
        return hipErrorOutOfMemory;
    }
    void* q = mmap(nullptr, n ? n : 1, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (q == MAP_FAILED) return hipErrorOutOfMemory;
    blocks[q] = n ? n : 1;
    if (device) {
        used += n;
        peak = used > peak ? used : peak;
        note("malloc " + std::to_string(n));
    }
    *p = q;
    return hipSuccess;
}

hipError_t release(void* p, bool device)
{
    if (!p) return hipSuccess;
    size_t n;
    {
        std::lock_guard<std::mutex> lk(mu);
        auto it = blocks.find(p);
        if (it == blocks.end()) return hipErrorInvalidValue;
        n = it->second;
        blocks.erase(it);
        if (device) {
            used -= n;
            note("free " + std::to_string(n));
        }
        munmap(p, n);
    }
    if (device && on_free && n >= on_free_bytes) on_free();
    return hipSuccess;
}

}  // namespace

extern "C" {

// ---- controls of a test ----
void host_hip_limit(size_t bytes) { limit = bytes; }
size_t host_hip_used() { std::lock_guard<std::mutex> lk(mu); return used; }
size_t host_hip_peak() { std::lock_guard<std::mutex> lk(mu); return peak; }
void host_hip_reset_peak() { std::lock_guard<std::mutex> lk(mu); peak = used; }
// fn is called after a device block of at least `bytes` has been freed
void host_hip_on_free(void (*fn)(), size_t bytes) { on_free = fn; on_free_bytes = bytes; }
// Untimed events recorded from now on stay unfinished until they are released
// one by one, in the order of their recording.
void host_hip_hold(int on) { std::lock_guard<std::mutex> lk(mu); hold = on != 0; }
int host_hip_held() { std::lock_guard<std::mutex> lk(mu); return (int)held.size(); }
int host_hip_release()
{
    std::lock_guard<std::mutex> lk(mu);
    if (held.empty()) return 0;
    held.front()->done = true;
    held.pop_front();
    return 1;
}
unsigned host_hip_launches(const char* part)
{
    std::lock_guard<std::mutex> lk(mu);
    unsigned n = 0;
    for (auto& k : launches)
        if (k.first.find(part) != std::string::npos) n += k.second;
    return n;
}
// Calls so far, a line each; clears them.  Returns the length.
size_t host_hip_log(char* out, size_t cap)
{
    std::lock_guard<std::mutex> lk(mu);
    const size_t n = log_text.size();
    if (out && cap > n) {
        std::memcpy(out, log_text.c_str(), n + 1);
        log_text.clear();
    }
    return n;
}

// ---- the runtime ----
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int)
{
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    p->totalGlobalMem = (size_t)288 << 30;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* s) { *p = const_cast<void*>(s); return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "host_hip error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }

hipError_t hipMalloc(void** p, size_t n) { return alloc(p, n, true); }
hipError_t hipFree(void* p) { return release(p, true); }
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t) { return alloc(p, n, true); }
hipError_t hipFreeAsync(void* p, hipStream_t) { return release(p, true); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return alloc(p, n, false); }
hipError_t hipHostFree(void* p) { return release(p, false); }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t)
{
    std::memset(d, v, n);
    return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t) new int; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { delete (int*)s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }

hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned flags)
{
    *e = (hipEvent_t) new Ev{!(flags & hipEventDisableTiming)};
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e)
{
    std::lock_guard<std::mutex> lk(mu);
    held.erase(std::remove(held.begin(), held.end(), (Ev*)e), held.end());
    delete (Ev*)e;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t)
{
    std::lock_guard<std::mutex> lk(mu);
    note("record");
    Ev* v = (Ev*)e;
    v->done = v->timed || !hold;
    if (!v->done) held.push_back(v);
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e)
{
    std::lock_guard<std::mutex> lk(mu);
    return ((Ev*)e)->done ? hipSuccess : hipErrorNotReady;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 2; return hipSuccess; }

hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, hipStream_t)
{
    std::lock_guard<std::mutex> lk(mu);
    const std::string& name = kernels[f];
    launches[name]++;
    note("launch " + name);
    return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* sh, hipStream_t* st)
{
    *g = *b = dim3(1);
    *sh = 0;
    *st = nullptr;
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) { static void* h = nullptr; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*)
{
    std::lock_guard<std::mutex> lk(mu);
    kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}

}  // extern "C"
