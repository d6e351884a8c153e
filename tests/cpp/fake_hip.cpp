// A HIP runtime without a device: memory is the host's, kernels are written down instead of run.  Loaded before a library of this
// repository (tests/fake_hip.py), it shows what the host code launches, captures and asks for.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

struct Dim
{
    unsigned x, y, z;
};
struct Graph
{
    int kernels;
};

namespace
{
    std::map<const void *, std::string> names;
    std::string text;
    Dim grid, block;
    size_t shared;
    void *on;
    Graph *capturing = nullptr;
    int largest = 1 << 30; // kernels of a graph that can be instantiated

    int note(const char *what, const std::string &rest)
    {
        text += std::string(what) + " " + rest + "\n";
        return 0;
    }
    std::string name(const void *f) { return names.count(f) ? names[f] : "?"; }
} // namespace

extern "C"
{
    const char *fake_hip_log() { return text.c_str(); }
    void fake_hip_clear() { text.clear(); }
    void fake_hip_largest_graph(int kernels) { largest = kernels; }

    void **__hipRegisterFatBinary(const void *)
    {
        static void *module;
        return &module;
    }
    void __hipUnregisterFatBinary(void **) {}
    void __hipRegisterFunction(void **, const void *f, char *, const char *device, unsigned, void *, void *, void *, void *, int *) { names[f] = device; }
    void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
    int __hipPushCallConfiguration(Dim g, Dim b, size_t bytes, void *stream)
    {
        grid = g, block = b, shared = bytes, on = stream;
        return 0;
    }
    int __hipPopCallConfiguration(Dim *g, Dim *b, size_t *bytes, void **stream)
    {
        *g = grid, *b = block, *bytes = shared, *stream = on;
        return 0;
    }
    int hipLaunchKernel(const void *f, Dim g, Dim b, void **, size_t bytes, void *)
    {
        if (capturing)
            ++capturing->kernels;
        char sizes[128];
        snprintf(sizes, sizeof(sizes), " %u %u %u %u %zu", g.x, g.y, g.z, b.x, bytes);
        return note(capturing ? "captured" : "launch", name(f) + sizes);
    }
    int hipFuncSetAttribute(const void *f, int, int value) { return note("lds", name(f) + " " + std::to_string(value)); }
    int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { return *n = 2, 0; }
    int hipGetSymbolAddress(void **p, const void *) { return *p = calloc(1, 64), 0; }

    int hipDeviceGetAttribute(int *v, int, int) { return *v = 256, 0; } // (compute units are all that is asked for)
    int hipGetDeviceCount(int *n) { return *n = 1, 0; }
    int hipGetDevice(int *d) { return *d = 0, 0; }
    int hipSetDevice(int) { return 0; }
    int hipDeviceSynchronize() { return 0; }
    const char *hipGetErrorString(int) { return "refused"; }
    int hipGetLastError() { return 0; }

    int hipMalloc(void **p, size_t n) { return *p = aligned_alloc(256, (n + 511) / 256 * 256), memset(*p, 0, n), 0; }
    int hipFree(void *p) { return free(p), 0; }
    int hipHostMalloc(void **p, size_t n, unsigned) { return hipMalloc(p, n); }
    int hipHostFree(void *p) { return hipFree(p); }
    int hipMemcpy(void *to, const void *from, size_t n, int) { return memcpy(to, from, n), 0; }
    int hipMemcpyAsync(void *to, const void *from, size_t n, int, void *) { return memcpy(to, from, n), 0; }
    int hipMemcpy2DAsync(void *to, size_t tp, const void *from, size_t fp, size_t w, size_t h, int, void *)
    {
        for (size_t i = 0; i < h; ++i)
            memcpy((char *)to + i * tp, (const char *)from + i * fp, w);
        return 0;
    }

    int hipStreamCreateWithFlags(void **s, unsigned) { return *s = malloc(1), 0; }
    int hipStreamDestroy(void *s) { return free(s), 0; }
    int hipStreamSynchronize(void *) { return 0; }
    int hipEventCreate(void **e) { return *e = malloc(1), 0; }
    int hipEventDestroy(void *e) { return free(e), 0; }
    int hipEventRecord(void *, void *) { return 0; }
    int hipEventElapsedTime(float *ms, void *, void *) { return *ms = 1.0f, 0; }

    int hipStreamBeginCapture(void *, int) { return capturing = new Graph{0}, note("begin", ""); }
    int hipStreamEndCapture(void *, Graph **g) { return *g = capturing, capturing = nullptr, note("end", std::to_string((*g)->kernels)); }
    int hipGraphDestroy(Graph *g) { return delete g, note("destroy", ""); }
    int hipGraphInstantiate(Graph **e, Graph *g, void *, char *, size_t)
    {
        if (g->kernels > largest)
            return 2; // hipErrorOutOfMemory
        return *e = new Graph(*g), note("instantiate", std::to_string(g->kernels));
    }
    int hipGraphLaunch(Graph *e, void *) { return note("replay", std::to_string(e->kernels)); }
    int hipGraphExecDestroy(Graph *e) { return delete e, 0; }
}
