// A HIP runtime without a device, for tests of the library's host code on the CPU: memory is the host's, streams and events
// are names, copies happen at once, and kernels do nothing but what stands below.  Loaded before libosph_gpu.so it takes
// the place of libamdhip64.  The test steers it through the stub_* functions.
#include <atomic>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <dlfcn.h>
#include <map>
#include <mutex>
#include <new>
#include <string>

namespace {

enum Error { SUCCESS = 0, INVALID = 1, OUT_OF_MEMORY = 2 };
enum MemoryType { UNREGISTERED = 0, HOST = 1, DEVICE = 2 };

std::mutex lock;
std::map<uintptr_t, std::pair<size_t, int>> blocks;  // address -> bytes, type
std::map<const void*, std::string> kernels;
std::string failing;            // launches of a kernel whose name holds this fail ...
int failures = 0;               // ... this many times
bool host_malloc_fails = false;
std::atomic<bool> new_fails{ false };
long long counters[10];          // see stub_counter
thread_local int device = 0, last_error = SUCCESS;
thread_local size_t launch_config[4];

struct Event { int device; };

int fail(int e) { return last_error = e; }

int type_of(const void* p) {
    const uintptr_t a = reinterpret_cast<uintptr_t>(p);
    auto it = blocks.upper_bound(a);
    if (it == blocks.begin()) return UNREGISTERED;
    --it;
    return a < it->first + it->second.first ? it->second.second : UNREGISTERED;
}

int allocate(void** p, size_t bytes, int type) {
    std::lock_guard<std::mutex> g(lock);
    *p = std::calloc(1, bytes + 64);
    if (!*p) return fail(OUT_OF_MEMORY);
    blocks[reinterpret_cast<uintptr_t>(*p)] = { bytes, type };
    return SUCCESS;
}

int release(void* p) {
    std::lock_guard<std::mutex> g(lock);
    if (p) blocks.erase(reinterpret_cast<uintptr_t>(p));
    std::free(p);
    return SUCCESS;
}

uint64_t ordered(double v) {
    uint64_t b;
    std::memcpy(&b, &v, 8);
    return b >> 63 ? ~b : b | 0x8000000000000000ull;
}

double box = 10.0;  // the particles' box, as the bounds kernels report it

void write_bounds(uint64_t* a) {  // min x, y, z, max x, y, z, max h, min h
    for (int k = 0; k < 3; ++k) a[k] = ordered(0.0), a[3 + k] = ordered(box);
    a[6] = a[7] = ordered(1.0);
}

template <typename T>
T arg(void** args, int k) {
    return *static_cast<T*>(args[k]);
}

void run(const std::string& name, void** args) {
    auto is = [&](const char* k) { return name.find(k) != std::string::npos; };
    if (is("6k_post")) {
        auto* src = arg<const uint64_t*>(args, 0);
        std::memcpy(arg<uint64_t*>(args, 2), src, 8 * arg<size_t>(args, 1));
        *arg<uint64_t*>(args, 3) = arg<uint64_t>(args, 4);
    } else if (is("10k_fill_u32E")) {
        for (size_t k = 0; k < arg<size_t>(args, 1); ++k) arg<uint32_t*>(args, 0)[k] = arg<uint32_t>(args, 2);
    } else if (is("8k_boundsE")) {
        write_bounds(arg<uint64_t*>(args, 1));
    } else if (is("9k_bounds3E")) {
        write_bounds(arg<uint64_t*>(args, 1));
    } else if (is("8k_levelsE")) {  // the host's words come by value: (host, posts, value)
        struct Post { uint64_t *host, *posts, value; };
        const Post post = arg<Post>(args, 4);
        post.host[7] = 1;
        *post.posts = post.value;
    } else if (is("14k_bounds_finalE")) {
        auto* small = arg<uint64_t*>(args, 2);  // the step's accumulators, the first class's bounds from word 16 on
        std::memset(small, 0, 8 * 64);
        write_bounds(small + 16);
        small[16 + 8] = 64;
        for (int k = 56; k < 62; ++k) small[k] = ordered(0.0);  // velocities
    } else if (is("13k_row_scatter")) {  // (where, row_start, first, row_count, slots, ...)
        std::memset(arg<uint32_t*>(args, 3), 0, 4 * size_t(arg<uint32_t>(args, 4)));
        ++counters[5];
    } else if (is("11k_row_count")) {  // (DevState, Grid, row_count, ...): the counts have to start at zero
        auto* counts = arg<uint32_t*>(args, 2);
        for (int k = 0; k < 4096; ++k) counters[4] += counts[k] != 0;
        counts[0] += 64;
    }
}

}  // namespace

void* operator new(size_t n) {
    if (new_fails) throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

extern "C" {

// ---- the test's side ------------------------------------------------------------------------------------------
// 0 copies to unregistered host memory, 1 to pinned host memory, 2 pinned allocations, 3 bytes of the largest copy to
// the host, 4 row counts found non-zero, 5 scatters, 6 events recorded on another device than their own, 7 the largest
// y or z extent of a launch, 8 launches of a search's, the pair sums' and gravity's kernels with an error pending,
// 9 launches for all members of a batch
long long stub_counter(int k) { return counters[k]; }
void stub_reset() { std::memset(counters, 0, sizeof(counters)); }
void stub_fail_kernel(const char* name, int times) { failing = name, failures = times; }
void stub_fail_host_malloc(int on) { host_malloc_fails = on != 0; }
void stub_fail_new(int on) { new_fails = on != 0; }
void stub_box(double size) { box = size; }

// ---- the library's side ---------------------------------------------------------------------------------------
int hipMalloc(void** p, size_t n) { return allocate(p, n, DEVICE); }
int hipFree(void* p) { return release(p); }
int hipHostMalloc(void** p, size_t n, unsigned) {
    if (host_malloc_fails) return fail(OUT_OF_MEMORY);
    ++counters[2];
    return allocate(p, n, HOST);
}
int hipHostFree(void* p) { return release(p); }
int hipPointerGetAttributes(int* attributes, const void* p) {  // hipPointerAttribute_t starts with the type
    std::lock_guard<std::mutex> g(lock);
    *attributes = type_of(p);
    return SUCCESS;
}
int hipMemcpy(void* dst, const void* src, size_t n, int) {
    std::memcpy(dst, src, n);
    return SUCCESS;
}
int hipMemcpyAsync(void* dst, const void* src, size_t n, int kind, void*) {
    if (kind == 2) {  // device to host
        std::lock_guard<std::mutex> g(lock);
        ++counters[type_of(dst) == UNREGISTERED ? 0 : 1];
        if (counters[3] < (long long)n) counters[3] = (long long)n;
    }
    std::memcpy(dst, src, n);
    return SUCCESS;
}
int hipMemset(void* p, int v, size_t n) {
    std::memset(p, v, n);
    return SUCCESS;
}
int hipMemsetAsync(void* p, int v, size_t n, void*) { return hipMemset(p, v, n); }
int hipGetDevice(int* d) {
    *d = device;
    return SUCCESS;
}
int hipSetDevice(int d) {
    device = d;
    return SUCCESS;
}
int hipGetLastError() {
    const int e = last_error;
    last_error = SUCCESS;
    return e;
}
int hipPeekAtLastError() { return last_error; }
const char* hipGetErrorString(int) { return "stub error"; }
int hipStreamCreateWithFlags(void** s, unsigned) {
    *s = std::malloc(8);
    return SUCCESS;
}
int hipStreamDestroy(void* s) {
    std::free(s);
    return SUCCESS;
}
int hipStreamSynchronize(void*) { return SUCCESS; }
int hipStreamQuery(void*) { return SUCCESS; }
int hipStreamWaitEvent(void*, void*, unsigned) { return SUCCESS; }
int hipStreamBeginCapture(void*, int) { return SUCCESS; }
int hipStreamEndCapture(void*, void** g) {
    *g = nullptr;
    return SUCCESS;
}
int hipGetStreamDeviceId(void*) { return device; }
int hipGraphInstantiate(void** e, void*, void*, char*, size_t) {
    *e = std::malloc(8);
    return SUCCESS;
}
int hipGraphLaunch(void*, void*) { return SUCCESS; }
int hipGraphExecDestroy(void* e) {
    std::free(e);
    return SUCCESS;
}
int hipGraphDestroy(void*) { return SUCCESS; }
int hipEventCreateWithFlags(void** e, unsigned) {
    *e = new (std::malloc(sizeof(Event))) Event{ device };
    return SUCCESS;
}
int hipEventCreate(void** e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void* e) {
    std::free(e);
    return SUCCESS;
}
int hipEventRecord(void* e, void*) {
    if (static_cast<Event*>(e)->device != device) ++counters[6];
    return SUCCESS;
}
int hipEventSynchronize(void*) { return SUCCESS; }
int hipEventElapsedTime(float* ms, void*, void*) {
    *ms = 1.0f;
    return SUCCESS;
}
int hipDeviceGetAttribute(int* v, int, int) {
    *v = 1;
    return SUCCESS;
}
int hipGetDevicePropertiesR0600(void*, int) { return SUCCESS; }
int hipGetSymbolAddress(void** p, const void*) {
    static char symbol[1 << 16];
    *p = symbol;
    return SUCCESS;
}
void** __hipRegisterFatBinary(const void*) {
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    kernels[host] = name;
}
struct Dim3 { uint32_t x, y, z; };
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shared, void* stream) {
    launch_config[0] = grid.x | uint64_t(grid.y) << 32;
    launch_config[1] = grid.z | uint64_t(block.x) << 32;
    launch_config[2] = shared;
    launch_config[3] = reinterpret_cast<size_t>(stream);
    return SUCCESS;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* shared, void** stream) {
    *grid = { uint32_t(launch_config[0]), uint32_t(launch_config[0] >> 32), uint32_t(launch_config[1]) };
    *block = { uint32_t(launch_config[1] >> 32), 1, 1 };
    *shared = launch_config[2];
    *stream = reinterpret_cast<void*>(launch_config[3]);
    return SUCCESS;
}
int hipLaunchKernel(const void* host, Dim3 grid, Dim3, void** args, size_t, void*) {
    const std::string& name = kernels[host];
    if (counters[7] < (long long)grid.y) counters[7] = grid.y;
    if (counters[7] < (long long)grid.z) counters[7] = grid.z;
    if (name.find("kb_") != std::string::npos) ++counters[9];
    for (const char* k : { "k_row_", "k_cell_", "kb_row_", "kb_cell_", "k_pack", "k_permute", "k_neighbor_lists", "k_pairs", "kb_pack",
                           "kb_permute", "kb_pairs", "kb_finalize",
                           "k_levels", "k_leaf_moments", "k_bucket", "k_moments_", "k_walk", "k_eval" }) {
        if (last_error != SUCCESS && name.find(k) != std::string::npos) ++counters[8];
    }
    if (failures > 0 && name.find(failing) != std::string::npos) {
        --failures;
        return fail(OUT_OF_MEMORY);
    }
    run(name, args);
    return SUCCESS;
}
}
