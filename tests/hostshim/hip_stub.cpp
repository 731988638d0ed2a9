// Stand-in for the HIP runtime on a machine without a GPU, so that the host
// paths of libzfv.so (allocations, copies, launches, error handling) run on the
// CPU: device memory is host memory with its extent remembered, copies are
// checked against it as the runtime checks them, kernels are recorded and not
// executed, and any call can be made to fail.  Loaded with global symbols before
// libzfv.so (tests/test_host_paths_cpu.py).
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include <hip/hip_runtime_api.h>

namespace {

struct Block {
    size_t size;
    bool device;
};
std::map<uintptr_t, Block> blocks;
std::map<const void*, std::string> kernels;
struct Launch {
    std::string name;
    uint64_t word;
};
std::vector<Launch> launches;
std::map<std::string, int> keep;   // part of a kernel's name -> the argument whose first word is kept
std::string fail_call;
int fail_after = 0;
hipError_t last_error = hipSuccess;
size_t pinned_bytes = 0;
std::map<std::string, float> cost;   // part of a kernel's name -> ms a launch takes (others 1)
float clock_ms = 0.0f;
int copies = 0;
std::map<hipEvent_t, float> events;

// the block that holds p, or null
const std::pair<const uintptr_t, Block>* block_of(const void* p) {
    auto it = blocks.upper_bound((uintptr_t)p);
    if (it == blocks.begin()) return nullptr;
    --it;
    return (uintptr_t)p < it->first + it->second.size ? &*it : nullptr;
}
bool fits(const void* p, size_t bytes) {
    const auto* b = block_of(p);
    return !b || (uintptr_t)p + bytes <= b->first + b->second.size;
}
// counts a call; true when it is the one that has to fail
bool fails(const std::string& call) {
    if (fail_call.empty() || call.find(fail_call) == std::string::npos || fail_after-- > 0) return false;
    fail_call.clear();
    return true;
}
hipError_t take(void** p, size_t bytes, bool device) {
    *p = calloc(1, bytes ? bytes : 1);
    if (!*p) return hipErrorOutOfMemory;
    blocks[(uintptr_t)*p] = Block{bytes, device};
    return hipSuccess;
}
hipError_t give(void* p) {
    if (!p) return hipSuccess;
    if (!blocks.erase((uintptr_t)p)) return hipErrorInvalidValue;
    free(p);
    return hipSuccess;
}
hipError_t copy(void* d, const void* s, size_t bytes) {
    if (!fits(d, bytes) || !fits(s, bytes)) return hipErrorInvalidValue;
    ++copies;
    memmove(d, s, bytes);
    return hipSuccess;
}
hipError_t ok(const char* call) { return fails(call) ? hipErrorUnknown : hipSuccess; }

}  // namespace

extern "C" {

// ---- what the tests read and set
// A runtime call by its name, or a launch by a part of the kernel's mangled
// name, fails once, after `after` successes.
void stub_fail(const char* call, int after) {
    fail_call = call;
    fail_after = after;
}
// The launches since the last reset: mangled names, and the 64-bit word that
// argument k begins with where stub_keep asked for it.
void stub_reset() { launches.clear(); }
int stub_launches() { return (int)launches.size(); }
const char* stub_launch(int i) { return launches[i].name.c_str(); }
void stub_keep(const char* kernel, int k) { keep[kernel] = k; }
uint64_t stub_word(int i) { return launches[i].word; }
size_t stub_pinned() { return pinned_bytes; }
int stub_copies() { return copies; }   // copies that went through the runtime so far
void stub_cost(const char* kernel, double ms) { cost[kernel] = (float)ms; }

// ---- registration and launches
void** __hipRegisterFatBinary(const void*) {
    static void* m = nullptr;
    return &m;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*,
                           int*) {
    kernels[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
static dim3 cfg_grid, cfg_block;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t) {
    cfg_grid = g;
    cfg_block = b;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) {
    *g = cfg_grid;
    *b = cfg_block;
    *m = 0;
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t) {
    Launch l{kernels[f], 0};
    if (fails(l.name)) return last_error = hipErrorLaunchFailure;
    for (const auto& kv : keep)
        if (l.name.find(kv.first) != std::string::npos) memcpy(&l.word, args[kv.second], sizeof(l.word));
    launches.push_back(l);
    float ms = 1.0f;
    for (const auto& kv : cost)
        if (l.name.find(kv.first) != std::string::npos) ms = kv.second;
    clock_ms += ms;
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = last_error;
    last_error = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "stub"; }

// ---- memory
hipError_t hipMalloc(void** p, size_t n) { return fails("hipMalloc") ? hipErrorOutOfMemory : take(p, n, true); }
hipError_t hipFree(void* p) { return give(p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (fails("hipHostMalloc")) return hipErrorOutOfMemory;
    pinned_bytes += n;
    return take(p, n, false);
}
hipError_t hipHostFree(void* p) {
    if (p) pinned_bytes -= blocks[(uintptr_t)p].size;
    return give(p);
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return copy(d, s, n); }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { return copy(d, s, n); }
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, hipMemcpyKind,
                            hipStream_t) {
    for (size_t i = 0; i < h; ++i)
        if (hipError_t e = copy((char*)d + i * dp, (const char*)s + i * sp, w)) return e;
    return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) {
    if (!fits(d, n)) return hipErrorInvalidValue;
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    const auto* b = block_of(p);
    memset(a, 0, sizeof(*a));
    if (!b) return hipErrorInvalidValue;
    a->type = b->second.device ? hipMemoryTypeDevice : hipMemoryTypeHost;
    a->devicePointer = const_cast<void*>(p);
    return hipSuccess;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t* base, size_t* size, hipDeviceptr_t p) {
    const auto* b = block_of(p);
    if (!b) return hipErrorNotFound;
    if (base) *base = (hipDeviceptr_t)b->first;
    if (size) *size = b->second.size;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static void* mem = calloc(1, (size_t)8 << 20);
    *p = mem;
    return hipSuccess;
}

// ---- devices, streams, events, graphs
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    memset(p, 0, sizeof(*p));
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    p->warpSize = 64;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
    *n = 1;
    return hipSuccess;
}
static int token;
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)&token; return ok("hipStreamCreateWithFlags"); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return ok("hipStreamSynchronize"); }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return ok("hipStreamWaitEvent"); }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)malloc(1); return ok("hipEventCreate"); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { events.erase(e); free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { events[e] = clock_ms; return ok("hipEventRecord"); }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) { *ms = events[b] - events[a]; return hipSuccess; }

}  // extern "C"
