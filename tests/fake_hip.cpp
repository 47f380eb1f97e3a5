// A HIP runtime without a GPU, for tests of the library's host code: it hands out addresses within a
// budget, copies between host memory and small allocations, and notes the kernels that would have been
// launched instead of running them. Loaded under the runtime's own library name before the library.
#include <hip/hip_runtime_api.h>

#include <sys/mman.h>
#include <unistd.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {
std::mutex m;
size_t budget = size_t(288) << 30, used = 0;
bool pinned_fails = false;
std::map<void*, size_t> pinned;  // and the bytes of all that were ever made
size_t pinned_live = 0, pinned_made = 0;
const void* shading_normals = nullptr;  // SceneDev::tri_vn of the last shading launch
bool freed = false;  // a kernel was given memory that is not allocated
int event_us = 0;  // a wait for an event takes that long
long mallocs_left = -1;  // hipMalloc fails from the one after these on (-1: never)
struct Block {
    size_t size, mapped;
};
std::map<char*, Block> blocks;                // device allocations
std::map<const void*, std::string> kernels;   // host stub -> device name
std::string log_;
constexpr size_t kBacked = size_t(64) << 20;  // larger allocations are addresses only

bool backed(const void* p)
{
    auto it = blocks.upper_bound(static_cast<char*>(const_cast<void*>(p)));
    if (it == blocks.begin()) return true;  // host memory
    --it;
    if (static_cast<const char*>(p) >= it->first + it->second.mapped) return true;
    return it->second.size <= kBacked;
}
thread_local hipError_t last = hipSuccess;
hipError_t failed(hipError_t e) { return last = e; }
bool live(const void* p)
{
    auto it = blocks.upper_bound(static_cast<char*>(const_cast<void*>(p)));
    return it != blocks.begin() && static_cast<const char*>(p) < (--it)->first + it->second.size;
}
thread_local struct {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
} config;
}  // namespace

extern "C" {
void fake_budget(size_t bytes) { budget = bytes; }
void fake_pinned_fails(int on) { pinned_fails = on != 0; }
void fake_mallocs_left(long n) { mallocs_left = n; }
size_t fake_used() { return used; }
size_t fake_pinned_live() { return pinned_live; }
size_t fake_pinned_made() { return pinned_made; }
const void* fake_shading_normals() { return shading_normals; }
int fake_freed() { return freed; }
void fake_event_us(int us) { event_us = us; }
const char* fake_log() { return log_.c_str(); }
void fake_clear() { log_.clear(); }

hipError_t hipMalloc(void** p, size_t n)
{
    std::lock_guard<std::mutex> lock(m);
    *p = nullptr;
    if (mallocs_left == 0 || used + n > budget) return failed(hipErrorOutOfMemory);
    if (mallocs_left > 0) --mallocs_left;
    const size_t mapped = (n + 4095) / 4096 * 4096 + 4096;
    void* a = mmap(nullptr, mapped, n <= kBacked ? PROT_READ | PROT_WRITE : PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (a == MAP_FAILED) return hipErrorOutOfMemory;
    blocks[static_cast<char*>(a)] = {n, mapped};
    used += n;
    *p = a;
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    std::lock_guard<std::mutex> lock(m);
    auto it = blocks.find(static_cast<char*>(p));
    if (it == blocks.end()) return p ? hipErrorInvalidValue : hipSuccess;
    munmap(p, it->second.mapped);
    used -= it->second.size;
    blocks.erase(it);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    std::lock_guard<std::mutex> lock(m);
    *p = pinned_fails ? nullptr : std::calloc(1, n);
    if (!*p) return failed(hipErrorOutOfMemory);
    pinned[*p] = n;
    pinned_live += n;
    pinned_made += n;
    return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
    std::lock_guard<std::mutex> lock(m);
    pinned_live -= pinned[p];
    pinned.erase(p);
    return std::free(p), hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) { return *f = budget - used, *t = budget, hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
    std::lock_guard<std::mutex> lock(m);
    if (backed(d) && backed(s)) std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t)
{
    std::lock_guard<std::mutex> lock(m);
    log_ += "memset\n";
    if (!live(d)) return failed(hipErrorInvalidValue);
    if (backed(d)) std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int)  // (the header renames it to its versioned name)
{
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError()
{
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipGetSymbolAddress(void** p, const void*)
{
    static char symbol[16 << 20];
    return *p = symbol, hipSuccess;
}
static hipError_t handle(void** h) { return *h = std::malloc(1), hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return handle(reinterpret_cast<void**>(e)); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return handle(reinterpret_cast<void**>(e)); }
hipError_t hipEventDestroy(hipEvent_t e) { return std::free(e), hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t)
{
    if (event_us) usleep(useconds_t(event_us));
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return handle(reinterpret_cast<void**>(s)); }
hipError_t hipStreamDestroy(hipStream_t s) { return std::free(s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t)
{
    if (event_us) usleep(useconds_t(event_us));
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return handle(reinterpret_cast<void**>(g)); }
hipError_t hipGraphDestroy(hipGraph_t g) { return std::free(g), hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t)
{
    return handle(reinterpret_cast<void**>(e));
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { return std::free(e), hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }

// a line per launch: the kernel's mangled name and, for the closest-hit launches of a bounce, their last
// argument (buffer and flags)
static hipError_t launched(const void* f, void** args)
{
    std::lock_guard<std::mutex> lock(m);
    const std::string& name = kernels[f];
    log_ += name;
    // the buffers that the first and the last kernel of a render get
    if ((name.find("set_wave_kernel") != std::string::npos || name.find("read_counters_kernel") != std::string::npos) &&
        !live(*static_cast<void**>(args[0])))
        freed = true;
    if (name.find("extend_kernel") != std::string::npos) log_ += " " + std::to_string(*static_cast<int*>(args[3]));
    log_ += "\n";
    if (name.find("shade_kernel") != std::string::npos || name.find("path_kernel") != std::string::npos)
        shading_normals = static_cast<const void**>(args[0])[4];
    // the first sample outside the film: none
    if (name.find("samples_begin_kernel") != std::string::npos) **static_cast<uint32_t**>(args[0]) = 0xFFFFFFFFu;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t) { return launched(f, args); }
hipError_t hipExtLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t, hipEvent_t, hipEvent_t, int)
{
    return launched(f, args);
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s)
{
    config = {grid, block, lds, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s)
{
    *grid = config.grid, *block = config.block, *lds = config.lds, *s = config.stream;
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void*)
{
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* stub, char*, const char* name, unsigned, void*, void*, void*, void*, int*)
{
    kernels[stub] = name;
}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
}
