// A HIP runtime without a device, preloaded in front of the real one by tests/test_cpu_host_rules.py: device memory is host
// memory under a byte budget, kernels do not run (their names are logged), every wait is over at once.  What the library
// decides on the host -- which kernel a call takes, what it allocates, what it refuses -- can be read off without a GPU.
#include <hip/hip_runtime_api.h>

#include <cmath>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

#define FAKE extern "C" __attribute__((visibility("default")))

namespace {
size_t g_budget = (size_t)1 << 40, g_used = 0;
bool g_capturing = false, g_sync_fails = false;
std::map<void *, size_t> g_blocks;
// (function statics: the library registers its kernels before this file's globals are made)
std::map<const void *, std::string> &names()
{
    static std::map<const void *, std::string> m;
    return m;
}
std::string &launch_log()
{
    static std::string s;
    return s;
}
long long *g_words;  // the pinned words that the library's set-up kernels leave their results in: here the test does
hipError_t g_last = hipSuccess;
hipError_t result(hipError_t e)
{
    if (e != hipSuccess) g_last = e;
    return e;
}
dim3 g_grid, g_block;
size_t g_shared;
double g_degree_first, g_degree_power;
int g_cells, g_cell_edges, g_twice;
hipStream_t g_stream;
}  // namespace

FAKE void fake_budget(size_t bytes) { g_budget = bytes; }
FAKE size_t fake_used() { return g_used; }
FAKE void fake_capturing(int on) { g_capturing = on != 0; }
FAKE void fake_sync_fails(int on) { g_sync_fails = on != 0; }
FAKE const char *fake_launches() { return launch_log().c_str(); }
FAKE void fake_word(int i, long long v) { g_words[i] = v; }
FAKE void fake_clear() { launch_log().clear(); }

FAKE void **__hipRegisterFatBinary(const void *)
{
    static void *handle;
    return &handle;
}
FAKE void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, uint3 *, uint3 *, dim3 *, dim3 *, int *) { names()[host] = name; }
FAKE void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
FAKE void __hipUnregisterFatBinary(void **) {}
FAKE hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream)
{
    g_grid = grid;
    g_block = block;
    g_shared = shared;
    g_stream = stream;
    return hipSuccess;
}
FAKE hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream)
{
    *grid = g_grid;
    *block = g_block;
    *shared = g_shared;
    *stream = g_stream;
    return hipSuccess;
}
// Two kernels whose results decide what the library does next are stood in for: the degree profile (sums of 64 degrees, falling as a
// power of their rank) and the edges of the dense cells (the first so many hold the same number, the others none).
FAKE void fake_degrees(double first, double power)
{
    g_degree_first = first;
    g_degree_power = power;
}
FAKE void fake_cells(int cells, int edges, int twice)
{
    g_cells = cells;
    g_cell_edges = edges;
    g_twice = twice;
}
FAKE hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3, void **args, size_t, hipStream_t)
{
    const std::string &name = names()[f];
    launch_log() += name + " " + std::to_string(grid.x) + "\n";
    if (name.find("k_slice_sums") != std::string::npos) {  // (sorted, rows, slices, sums)
        float *const sums = *static_cast<float **>(args[3]);
        for (int s = 0; s < *static_cast<int *>(args[2]); ++s) sums[s] = (float)(g_degree_first * std::pow(s + 1.0, -g_degree_power));
    } else if (name.find("k_cells_count") != std::string::npos) {  // (ptr, col, rank, sorted, ranked, rows, lb, ntiles, cnt, twice)
        int *const cnt = *static_cast<int **>(args[8]);
        for (int c = 0; c < g_cells; ++c) cnt[2 * c] = g_cell_edges;
        **static_cast<int **>(args[9]) = g_twice;
    }
    return hipSuccess;
}
FAKE hipError_t hipGetDeviceCount(int *n)
{
    *n = 1;
    return hipSuccess;
}
FAKE hipError_t hipGetDevice(int *d)
{
    *d = 0;
    return hipSuccess;
}
FAKE int hipGetStreamDeviceId(hipStream_t) { return 0; }
FAKE hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    *s = nullptr;
    return hipSuccess;
}
FAKE hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    *e = nullptr;
    return hipSuccess;
}
FAKE hipError_t hipSetDevice(int) { return hipSuccess; }
FAKE hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    memset(p, 0, sizeof(*p));
    strcpy(p->name, "none");
    strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
FAKE hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int)
{
    *v = 0;
    return hipSuccess;
}
FAKE hipError_t hipMalloc(void **p, size_t bytes)
{
    *p = nullptr;
    if (bytes > g_budget - g_used) return result(hipErrorOutOfMemory);
    *p = aligned_alloc(256, (bytes + 255) & ~(size_t)255);
    if (!*p) return result(hipErrorOutOfMemory);
    memset(*p, 0, bytes);  // (what no kernel writes)
    g_blocks[*p] = bytes;
    g_used += bytes;
    return hipSuccess;
}
FAKE hipError_t hipFree(void *p)
{
    if (!p) return hipSuccess;
    const auto it = g_blocks.find(p);
    if (it == g_blocks.end()) return result(hipErrorInvalidValue);
    g_used -= it->second;
    g_blocks.erase(it);
    free(p);
    return hipSuccess;
}
FAKE hipError_t hipHostMalloc(void **p, size_t bytes, unsigned)
{
    *p = calloc(1, bytes);
    if (bytes == 512) g_words = static_cast<long long *>(*p);
    return hipSuccess;
}
FAKE hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
    memcpy(d, s, n);
    return hipSuccess;
}
FAKE hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    memcpy(d, s, n);
    return hipSuccess;
}
FAKE hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t)
{
    memset(d, v, n);
    return hipSuccess;
}
FAKE hipError_t hipGetSymbolAddress(void **p, const void *)
{
    static void *const q = aligned_alloc(256, 256);  // (no kernel runs: only the address is looked at)
    *p = q;
    return hipSuccess;
}
FAKE hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *st)
{
    *st = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
FAKE hipError_t hipGetLastError()
{
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
FAKE hipError_t hipDeviceSynchronize() { return g_sync_fails ? result(hipErrorStreamCaptureUnsupported) : hipSuccess; }
FAKE hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
FAKE hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
FAKE hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
FAKE hipError_t hipEventCreate(hipEvent_t *e)
{
    *e = nullptr;
    return hipSuccess;
}
FAKE hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
FAKE hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
FAKE hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)  // every measurement is faster than the one before: the last candidate wins
{
    static float t = 1e6f;
    *ms = t *= 0.99f;
    return hipSuccess;
}
FAKE hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
