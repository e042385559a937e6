// A HIP runtime that runs nothing: memory is host memory, a launch is written down (kernel, grid,
// block, dynamic LDS and the limit its function has been given).  Loaded with RTLD_GLOBAL before
// libpned_gpu.so it takes the place of the runtime, so the host side of a call (plans, tables,
// choice of kernel and launch shape) can be looked at without a GPU.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

struct Dim {
    uint32_t x, y, z;
};
static std::map<const void *, std::string> names;
static std::map<const void *, int> limits;
static std::string launches;
static std::map<std::string, float> costs;   // by part of the kernel's name
static float clock_ms;
static size_t uploaded;
static Dim cfg_grid, cfg_block;
static size_t cfg_lds;
static void *cfg_stream;
static char dummy[64];

static int alloc(void **p, size_t n)
{
    *p = calloc(1, n ? n : 1);   // (untouched pages of a large vector cost nothing)
    return *p ? 0 : 2;
}
static int copy(void *dst, const void *src, size_t n)
{
    memmove(dst, src, n);
    return 0;
}

extern "C" {

// the launches since the last call, one a line
const char *record_take()
{
    static std::string out;
    out.swap(launches);
    launches.clear();
    return out.c_str();
}

// bytes copied to the device so far
size_t record_uploaded() { return uploaded; }
// the time of a launch of a kernel whose name holds `part` (others 1 ms)
void record_cost(const char *part, float ms) { costs[part] = ms; }

void **__hipRegisterFatBinary(const void *) { return reinterpret_cast<void **>(dummy); }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *,
                           void *, int *)
{
    names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim grid, Dim block, size_t lds, void *stream)
{
    cfg_grid = grid;
    cfg_block = block;
    cfg_lds = lds;
    cfg_stream = stream;
    return 0;
}
int __hipPopCallConfiguration(Dim *grid, Dim *block, size_t *lds, void **stream)
{
    *grid = cfg_grid;
    *block = cfg_block;
    *lds = cfg_lds;
    *stream = cfg_stream;
    return 0;
}
int hipLaunchKernel(const void *f, Dim grid, Dim block, void **, size_t lds, void *)
{
    launches += names[f] + " " + std::to_string(grid.x) + " " + std::to_string(block.x) + " " + std::to_string(lds) +
                " " + std::to_string(limits[f]) + "\n";
    float ms = 1.0f;
    for (const auto &c : costs)
        if (names[f].find(c.first) != std::string::npos) ms = c.second;
    clock_ms += ms;
    return 0;
}
int hipFuncSetAttribute(const void *f, int, int value)
{
    limits[f] = value;
    return 0;
}
// LDS and wave slots of a CU (registers are not known here)
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int block, size_t lds)
{
    const size_t by_lds = 160 * 1024 / (lds ? lds : 1), by_waves = 2048 / block;
    *n = (int)(by_lds < by_waves ? by_lds : by_waves);
    return 0;
}
int hipDeviceGetAttribute(int *v, int, int) { return *v = 256, 0; }   // only asked for the compute units
int hipGetDeviceCount(int *n) { return *n = 1, 0; }
int hipGetDevice(int *d) { return *d = 0, 0; }
int hipSetDevice(int) { return 0; }
int hipGetLastError() { return 0; }
const char *hipGetErrorString(int) { return "no GPU here"; }
int hipGetSymbolAddress(void **p, const void *) { return *p = dummy, 0; }
int hipMalloc(void **p, size_t n) { return alloc(p, n); }
int hipMallocAsync(void **p, size_t n, void *) { return alloc(p, n); }
int hipHostMalloc(void **p, size_t n, unsigned) { return alloc(p, n); }
int hipFree(void *p) { return free(p), 0; }
int hipFreeAsync(void *p, void *) { return free(p), 0; }
int hipHostFree(void *p) { return free(p), 0; }
int hipMemcpy(void *dst, const void *src, size_t n, int kind)
{
    if (kind == 1) uploaded += n;
    return copy(dst, src, n);
}
int hipMemcpyAsync(void *dst, const void *src, size_t n, int kind, void *) { return hipMemcpy(dst, src, n, kind); }
int hipMemsetAsync(void *, int, size_t, void *) { return 0; }
int hipStreamCreateWithFlags(void **s, unsigned) { return *s = dummy, 0; }
int hipStreamDestroy(void *) { return 0; }
int hipStreamSynchronize(void *) { return 0; }
int hipStreamBeginCapture(void *, int) { return 0; }
int hipStreamEndCapture(void *, void **g) { return *g = dummy, 0; }
int hipGraphInstantiate(void **e, void *, void **, char *, size_t) { return *e = dummy, 0; }
int hipGraphLaunch(void *, void *) { return 0; }
int hipGraphDestroy(void *) { return 0; }
int hipGraphExecDestroy(void *) { return 0; }
int hipEventCreate(void **e) { return *e = calloc(1, sizeof(float)), 0; }
int hipEventDestroy(void *e) { return free(e), 0; }
int hipEventRecord(void *e, void *) { return *static_cast<float *>(e) = clock_ms, 0; }
int hipEventSynchronize(void *) { return 0; }
int hipEventElapsedTime(float *ms, void *a, void *b)
{
    return *ms = *static_cast<float *>(b) - *static_cast<float *>(a), 0;
}
}
