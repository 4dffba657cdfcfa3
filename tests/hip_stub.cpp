// A HIP runtime without a device: memory is the host's, kernels are recorded and
// not run, and a call can be told to fail.  The library's host paths (error
// paths, launch choices, which device a call is made on) run on it on any
// machine: loaded with RTLD_GLOBAL before libqpslice.so, its functions stand in
// for the runtime's.  Two devices; a graph is instantiated on the device of the
// stream it was captured on, as the runtime requires.
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
struct Stream { int device; bool capture; int syncs; };
struct Graph { int device; };
struct Launch { std::string name; size_t lds; long blocks; };
struct Config { dim3 grid, block; size_t lds; hipStream_t st; };

thread_local int cur = 0;
// never destroyed: the library is unloaded after this file's statics
auto &names = *new std::map<const void *, std::string>;
auto &granted = *new std::map<const void *, size_t>;
auto &vars = *new std::map<const void *, void *>;
auto &host_flags = *new std::map<void *, unsigned>;
auto &host_bytes = *new std::map<void *, size_t>;
auto &streams = *new std::vector<Stream *>;
auto &launches = *new std::vector<Launch>;
auto &words = *new std::map<std::string, unsigned long long>;   // k_push: its argument 1
thread_local std::vector<Config> configs;
int max_lds = 163840, cus = 256;
int fail_launch = 0;       // the graph launch (counted from now) that fails
int pageable = 0;          // copies to host memory that is not pinned
int graph_launches = 0, instantiations = 0;
size_t residual_bytes = 0; // a graph launch fills the host allocations of this size
double residual = 0.0;     // with this value
int key_changes = 0;       // what a beam push counts
}  // namespace

extern "C" {
// ---- what a test sets and reads ----
void stub_limits(int lds, int units) { max_lds = lds; cus = units; }
void stub_fail_launch(int n) { fail_launch = n; }
void stub_residual(size_t n, double v) { residual_bytes = n; residual = v; }
void stub_key_changes(int n) { key_changes = n; }
int stub_pageable() { return pageable; }
int stub_graph_launches() { return graph_launches; }
int stub_instantiations() { return instantiations; }
int stub_syncs(int stream) { return streams[stream]->syncs; }
int stub_streams() { return (int)streams.size(); }
void stub_clear_launches() { launches.clear(); }
int stub_launched(const char *part)
{
    int n = 0;
    for (const Launch &l : launches) n += l.name.find(part) != std::string::npos;
    return n;
}
// workgroups of the last such launch
long stub_blocks(const char *part)
{
    long v = -1;
    for (const Launch &l : launches)
        if (l.name.find(part) != std::string::npos) v = l.blocks;
    return v;
}
// LDS bytes of the last such launch
long stub_lds(const char *part)
{
    long v = -1;
    for (const Launch &l : launches)
        if (l.name.find(part) != std::string::npos) v = (long)l.lds;
    return v;
}
unsigned long long stub_word(const char *part)
{
    for (const auto &w : words)
        if (w.first.find(part) != std::string::npos) return w.second;
    return 0;
}
// the flags of the host allocation of n bytes made last; ~0: none
unsigned stub_host_flags(size_t n)
{
    unsigned f = ~0u;
    for (const auto &b : host_bytes)
        if (b.second == n) f = host_flags[b.first];
    return f;
}

// ---- the runtime ----
void **__hipRegisterFatBinary(const void *) { static void *m; return &m; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *fn, char *, const char *name, unsigned, void *,
                           void *, dim3 *, dim3 *, int *) { names[fn] = name; }
void __hipRegisterVar(void **, void *var, char *, char *, int, size_t n, int, int)
{
    vars[var] = std::calloc(1, n ? n : 1);
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t st)
{
    configs.push_back({g, b, lds, st});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *st)
{
    const Config c = configs.back();
    configs.pop_back();
    *g = c.grid; *b = c.block; *lds = c.lds; *st = c.st;
    return hipSuccess;
}
static thread_local hipError_t last = hipSuccess;
hipError_t hipLaunchKernel(const void *fn, dim3 g, dim3 b, void **args, size_t lds, hipStream_t)
{
    const size_t limit = granted.count(fn) ? granted[fn] : 65536;
    if (!g.x || !g.y || !g.z || !b.x || lds > limit || lds > (size_t)max_lds)
        return last = hipErrorInvalidConfiguration;
    launches.push_back({names[fn], lds, (long)g.x * g.y * g.z});
    if (names[fn].find("k_push") != std::string::npos)
        std::memcpy(&words[names[fn]], args[1], 8);
    if (names[fn].find("k_ctl_reset") != std::string::npos) {   // the host reads it back
        int *ctl = *static_cast<int **>(args[0]);
        ctl[0] = 1;
        ctl[1] = 0;
    }
    if (names[fn].find("k_permute") != std::string::npos && names[fn].find("PiS3_ji") != std::string::npos) {
        // a beam push: every particle lives, and this many places change cell
        **static_cast<int **>(args[6]) = (int)*static_cast<long long *>(args[0]);
        **static_cast<int **>(args[7]) = key_changes;
    }
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *fn, hipFuncAttribute, int v)
{
    if (v > max_lds) return last = hipErrorInvalidValue;
    granted[fn] = v;
    return hipSuccess;
}
hipError_t hipGetLastError() { const hipError_t e = last; last = hipSuccess; return e; }
const char *hipGetErrorString(hipError_t) { return "stub error"; }
hipError_t hipSetDevice(int d) { cur = d; return d >= 0 && d < 4 ? hipSuccess : hipErrorInvalidDevice; }
hipError_t hipGetDevice(int *d) { *d = cur; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int)
{
    *v = a == hipDeviceAttributeMaxSharedMemoryPerBlock ? max_lds
       : a == hipDeviceAttributeMultiprocessorCount     ? cus
       : a == hipDeviceAttributeWarpSize                ? 64 : 0;
    return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int)
{
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->gcnArchName, "gfx950:sramecc+:xnack-");
    p->warpSize = 64;
    p->multiProcessorCount = cus;
    p->maxThreadsPerBlock = 1024;
    p->sharedMemPerBlock = max_lds;
    p->maxGridSize[0] = 1 << 30;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *v) { *p = vars[v]; return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { *p = std::malloc(n); return *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned flags)
{
    *p = std::calloc(1, n);
    host_flags[*p] = flags;
    host_bytes[*p] = n;
    return hipSuccess;
}
hipError_t hipHostFree(void *p) { host_flags.erase(p); host_bytes.erase(p); std::free(p); return hipSuccess; }
static bool capturing(hipStream_t st) { return st && reinterpret_cast<Stream *>(st)->capture; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind kind, hipStream_t st)
{
    if (kind == hipMemcpyDeviceToHost && !host_bytes.count(d)) ++pageable;
    if (!capturing(st)) std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n) { std::memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st)
{
    if (!capturing(st)) std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *st, unsigned)
{
    streams.push_back(new Stream{cur, false, 0});
    *st = reinterpret_cast<hipStream_t>(streams.back());
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t st)
{
    if (st) ++reinterpret_cast<Stream *>(st)->syncs;
    return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
int hipGetStreamDeviceId(hipStream_t st) { return st ? reinterpret_cast<Stream *>(st)->device : cur; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = reinterpret_cast<hipEvent_t>(std::malloc(1)); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 0.f; return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t st, hipStreamCaptureMode)
{
    reinterpret_cast<Stream *>(st)->capture = true;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t st, hipGraph_t *g)
{
    Stream *s = reinterpret_cast<Stream *>(st);
    s->capture = false;
    *g = reinterpret_cast<hipGraph_t>(new Graph{s->device});
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *, char *, size_t)
{
    ++instantiations;
    if (reinterpret_cast<Graph *>(g)->device != cur) return hipErrorInvalidDevice;
    *e = reinterpret_cast<hipGraphExec_t>(new Graph(*reinterpret_cast<Graph *>(g)));
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t)
{
    ++graph_launches;
    if (fail_launch && --fail_launch == 0) return hipErrorLaunchFailure;
    if (residual_bytes)
        for (const auto &b : host_bytes)
            if (b.second == residual_bytes)
                for (size_t i = 0; i < b.second / 8; ++i) static_cast<double *>(b.first)[i] = residual;
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { delete reinterpret_cast<Graph *>(g); return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { delete reinterpret_cast<Graph *>(e); return hipSuccess; }
}
