// Stand-in for the HIP runtime in tests without a GPU: device memory is host memory, kernels
// are recorded and not run, and the source of every copy from host memory is compared, when
// its stream is waited for, with what it held when the copy was queued (a source that was
// freed or written before that wait is counted as stale).  Loaded with RTLD_GLOBAL before
// libdmftgpu.so, whose HIP calls then resolve here (tests/host_hip.py).
#include <cxxabi.h>
#include <sys/mman.h>
#include <sys/uio.h>
#include <unistd.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {

struct Dim3 {
    uint32_t x, y, z;
};
struct Pending {
    const void* src;
    std::vector<char> held;
    void* stream;
};
struct Config {
    Dim3 grid, block;
    size_t shm;
    void* stream;
};

std::map<const char*, size_t> blocks;  // device allocations
size_t in_use = 0, peak = 0;
std::vector<Pending> pending;
int stale = 0;
std::string events;
std::map<const void*, std::string> kernels;
std::vector<Config> configs;
char symbol[64];

bool on_device(const void* p)
{
    auto it = blocks.upper_bound((const char*)p);
    if (it == blocks.begin()) return false;
    --it;
    return (const char*)p < it->first + it->second;
}

void note(const char* fmt, const char* name, unsigned long long a = 0, unsigned long long b = 0, unsigned long long c = 0)
{
    char buf[1024];
    snprintf(buf, sizeof(buf), fmt, name, a, b, c);
    events += buf;
}

// stream null: every stream
void settle(void* stream, bool all)
{
    std::vector<Pending> left;
    for (auto& p : pending) {
        if (!all && p.stream != stream) {
            left.push_back(p);
            continue;
        }
        std::vector<char> now(p.held.size());
        iovec to{now.data(), now.size()}, from{const_cast<void*>(p.src), now.size()};  // the source may be unmapped by now
        if (process_vm_readv(getpid(), &to, 1, &from, 1, 0) != (ssize_t)now.size() || now != p.held) ++stale;
    }
    pending.swap(left);
}

int copy(void* dst, const void* src, size_t bytes, void* stream, bool async)
{
    const bool from_host = on_device(dst) && !on_device(src), to_host = !on_device(dst);
    note("copy %s %llu %llu\n", from_host ? "h2d" : to_host ? "d2h" : "d2d", bytes, (unsigned long long)(uintptr_t)stream);
    if (async && from_host) pending.push_back({src, std::vector<char>((const char*)src, (const char*)src + bytes), stream});
    if (bytes <= (64u << 20)) memmove(dst, src, bytes);
    return 0;
}

}  // namespace

extern "C" {

const char* host_hip_events() { return events.c_str(); }
int host_hip_stale()
{
    settle(nullptr, true);
    return stale;
}
size_t host_hip_peak() { return peak; }
void host_hip_reset()
{
    settle(nullptr, true);
    events.clear();
    stale = 0;
    peak = in_use;
}
void* host_hip_alloc(size_t bytes)
{
    if (!bytes) bytes = 1;
    // pages that nothing touches take no memory, so sizes of a GPU's memory can be asked for
    void* p = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (p == MAP_FAILED) return nullptr;
    blocks[(char*)p] = bytes;
    in_use += bytes;
    if (in_use > peak) peak = in_use;
    return p;
}

int hipMalloc(void** p, size_t bytes)
{
    note("malloc%s %llu\n", "", bytes);
    *p = host_hip_alloc(bytes);
    return *p ? 0 : 2;
}
int hipFree(void* p)
{
    settle(nullptr, true);
    auto it = blocks.find((const char*)p);
    if (it == blocks.end()) return p ? 1 : 0;
    in_use -= it->second;
    munmap(p, it->second);
    blocks.erase(it);
    return 0;
}
int hipMemcpy(void* dst, const void* src, size_t bytes, int) { return copy(dst, src, bytes, nullptr, false); }
int hipMemcpyAsync(void* dst, const void* src, size_t bytes, int, void* stream)
{
    return copy(dst, src, bytes, stream, true);
}

void** __hipRegisterFatBinary(const void*)
{
    static void* module = nullptr;
    return &module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*)
{
    int status = 0;
    char* d = abi::__cxa_demangle(name, nullptr, nullptr, &status);
    std::string s = status == 0 ? d : name;
    free(d);
    kernels[host] = s;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shm, void* stream)
{
    configs.push_back({grid, block, shm, stream});
    return 0;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* shm, void** stream)
{
    const Config c = configs.back();
    configs.pop_back();
    *grid = c.grid;
    *block = c.block;
    *shm = c.shm;
    *stream = c.stream;
    return 0;
}
int hipLaunchKernel(const void* f, Dim3 grid, Dim3 block, void**, size_t shm, void* stream)
{
    char buf[256];
    snprintf(buf, sizeof(buf), " | %u %u %u | %u %u %u | %zu | %llu\n", grid.x, grid.y, grid.z, block.x, block.y, block.z, shm,
             (unsigned long long)(uintptr_t)stream);
    events += "launch " + kernels[f] + buf;
    // what the runtime refuses
    return grid.x && grid.y && grid.z && grid.y <= 65535 && grid.z <= 65535 && block.x * block.y * block.z <= 1024 &&
                   shm <= 160 * 1024
               ? 0
               : 9;
}
int hipFuncSetAttribute(const void*, int, int) { return 0; }

int hipGetDevice(int* d)
{
    *d = 0;
    return 0;
}
const char* hipGetErrorString(int) { return "host_hip"; }
int hipGetLastError() { return 0; }
int hipGetSymbolAddress(void** p, const void*)
{
    *p = symbol;
    return 0;
}

int hipStreamCreateWithFlags(void** s, unsigned)
{
    *s = malloc(1);
    return 0;
}
int hipStreamDestroy(void* s)
{
    settle(s, false);
    free(s);
    return 0;
}
int hipStreamSynchronize(void* s)
{
    note("sync%s %llu\n", "", (unsigned long long)(uintptr_t)s);
    settle(s, false);
    return 0;
}
int hipStreamWaitEvent(void*, void*, unsigned) { return 0; }
int hipStreamBeginCapture(void*, int) { return 0; }
int hipStreamEndCapture(void*, void** g)
{
    *g = malloc(1);
    return 0;
}
int hipGraphInstantiate(void** e, void*, void**, char*, size_t)
{
    *e = malloc(1);
    return 0;
}
int hipGraphLaunch(void*, void*) { return 0; }
int hipGraphDestroy(void* g)
{
    free(g);
    return 0;
}
int hipGraphExecDestroy(void* g)
{
    free(g);
    return 0;
}
int hipEventCreate(void** e)
{
    *e = malloc(1);
    return 0;
}
int hipEventCreateWithFlags(void** e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void* e)
{
    free(e);
    return 0;
}
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*)
{
    settle(nullptr, true);
    return 0;
}
int hipEventElapsedTime(float* ms, void*, void*)
{
    *ms = 1.0f;
    return 0;
}

}  // extern "C"
