// The HIP runtime calls of libbelewitte_hip.so on host memory, for tests of
// its host code without a GPU: copies are copies, kernels are not run but
// listed, and an allocation can be made to fail.  Loaded (RTLD_GLOBAL) before
// the library, in a process of its own.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {

struct Dim3 {
    uint32_t x, y, z;
};
struct Config {
    Dim3 grid, block;
    size_t lds;
    void *stream;
} config;

std::map<const void *, std::string> kernels;
std::string calls;  // one line per launch, allocation and attribute set
int last = 0;
uint64_t fail_from = ~0ull;  // allocations of at least this many bytes fail
int64_t live = 0;

int record(int error)
{
    if (error) last = error;
    return error;
}

}  // namespace

extern "C" {

void fake_fail_from(uint64_t bytes) { fail_from = bytes; }
void fake_clear() { calls.clear(); }
const char *fake_calls() { return calls.c_str(); }
int64_t fake_live() { return live; }

int hipMalloc(void **p, size_t n)
{
    if (n >= fail_from) return record(2);  // hipErrorOutOfMemory
    calls += "alloc " + std::to_string(n) + "\n";
    live++;
    *p = std::calloc(1, n);
    return 0;
}
int hipFree(void *p)
{
    if (p) live--;
    std::free(p);
    return 0;
}
int hipHostMalloc(void **p, size_t n, unsigned) { return hipMalloc(p, n); }
int hipHostFree(void *p) { return hipFree(p); }
int hipMemcpy(void *d, const void *s, size_t n, int)
{
    std::memcpy(d, s, n);
    return 0;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *) { return hipMemcpy(d, s, n, k); }
int hipMemsetAsync(void *d, int v, size_t n, void *)
{
    std::memset(d, v, n);
    return 0;
}

int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t lds, void *stream)
{
    config = {grid, block, lds, stream};
    return 0;
}
int __hipPopCallConfiguration(Dim3 *grid, Dim3 *block, size_t *lds, void **stream)
{
    *grid = config.grid, *block = config.block, *lds = config.lds, *stream = config.stream;
    return 0;
}
int hipLaunchKernel(const void *f, Dim3 grid, Dim3 block, void **, size_t lds, void *)
{
    calls += "launch " + kernels[f] + " grid " + std::to_string(grid.x) + " block " + std::to_string(block.x) +
             " lds " + std::to_string(lds) + "\n";
    return last;  // a launch reports an error that was left behind
}
int hipFuncSetAttribute(const void *f, int, int value)
{
    calls += "attribute " + kernels[f] + " " + std::to_string(value) + "\n";
    return 0;
}
void **__hipRegisterFatBinary(const void *)
{
    static void *handle;
    return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *,
                           void *, int *)
{
    kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, const char *, int, size_t, int, int) {}

int hipGetLastError()
{
    const int e = last;
    last = 0;
    return e;
}
const char *hipGetErrorString(int) { return "fake error"; }
int hipGetDevice(int *d) { return *d = 0; }
int hipSetDevice(int) { return 0; }
int hipGetDeviceCount(int *n)
{
    *n = 1;
    return 0;
}
int hipDeviceGetAttribute(int *v, int, int)
{
    *v = 256;  // compute units; any positive clock rate
    return 0;
}
int hipDeviceSynchronize() { return 0; }
int hipStreamSynchronize(void *) { return 0; }
int hipStreamCreateWithFlags(void **s, unsigned) { return hipMalloc(s, 8); }
int hipStreamDestroy(void *s) { return hipFree(s); }
int hipEventCreate(void **e) { return hipMalloc(e, 8); }
int hipEventDestroy(void *e) { return hipFree(e); }
int hipEventRecord(void *, void *) { return 0; }
int hipEventSynchronize(void *) { return 0; }
int hipEventElapsedTime(float *ms, void *, void *)
{
    *ms = 0;
    return 0;
}

}  // extern "C"
