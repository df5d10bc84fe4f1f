// fake_hip.h -- the HIP calls libsolaris_amd.so makes, for host-side checks
// without a GPU: a program that includes this and is linked with -rdynamic
// takes the place of the HIP library for them.  Device memory is host memory,
// copies and fills happen at once, kernels do nothing but call a hook, and
// every call is counted.  What is queued on a stream counts as pending until a
// wait covers it, so a check can tell whether a call left work behind.
#pragma once

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <utility>
#include <vector>

#include <hip/hip_runtime_api.h>

struct ihipStream_t {
    long queued = 0, done = 0;
    std::vector<std::pair<ihipStream_t *, long>> waits;   // another stream's work that this one waits for
    bool capturing = false;
};
struct ihipEvent_t { ihipStream_t *stream = nullptr; long at = 0; };
struct ihipGraph { int kernels; };
struct hipGraphExec { int kernels; };

namespace fake {
inline std::map<std::string, long> &calls() { static std::map<std::string, long> m; return m; }
inline std::map<std::string, long> &kernels() { static std::map<std::string, long> m; return m; }   // launches by name
inline std::map<const void *, std::string> &names() { static std::map<const void *, std::string> m; return m; }
inline std::vector<ihipStream_t *> &streams() { static std::vector<ihipStream_t *> v; return v; }
inline int &device() { static int d = 0; return d; }               // the current device, of two
inline std::map<int, long> &made_on() { static std::map<int, long> m; return m; }   // allocations and streams by device
inline std::map<void *, size_t> &device_memory() { static std::map<void *, size_t> m; return m; }
inline std::function<void(const std::string &, void **)> &on_kernel()
{
    static std::function<void(const std::string &, void **)> f;
    return f;
}
inline std::function<void()> &on_graph() { static std::function<void()> f; return f; }
// the `fail_at`-th call (from 1) of `fail_name` fails; 0: none
inline std::string &fail_name() { static std::string s; return s; }
inline long &fail_at() { static long n = 0; return n; }
inline ihipStream_t *stream(hipStream_t s)
{
    static ihipStream_t null;
    return s ? s : &null;
}
inline bool fails(const char *name)
{
    ++calls()[name];
    return fail_at() > 0 && fail_name() == name && --fail_at() == 0;
}
inline void settle(ihipStream_t *s, long upto)
{
    if (upto > s->done) s->done = upto;
    for (auto &w : s->waits) if (w.second > w.first->done) w.first->done = w.second;
}
inline long pending()
{
    long n = 0;
    for (ihipStream_t *s : streams()) n += s->queued - s->done;
    return n;
}
inline void forget() { calls().clear(); kernels().clear(); made_on().clear(); }
struct Launch { dim3 grid, block; size_t lds; hipStream_t stream; };
inline std::vector<Launch> &pushed() { static std::vector<Launch> v; return v; }
}  // namespace fake

#define FAKE(name)                                                                                                     \
    do {                                                                                                               \
        if (fake::fails(name)) return hipErrorUnknown;                                                                 \
    } while (0)

extern "C" {
struct uint3_ { unsigned x, y, z; };
void **__hipRegisterFatBinary(const void *) { static void *p; return &p; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *)
{
    fake::names()[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s)
{
    fake::pushed().push_back({g, b, lds, s});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s)
{
    const fake::Launch l = fake::pushed().back();
    fake::pushed().pop_back();
    *g = l.grid; *b = l.block; *lds = l.lds; *s = l.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t s)
{
    FAKE("hipLaunchKernel");
    const std::string &name = fake::names()[f];
    ++fake::kernels()[name];
    ++fake::stream(s)->queued;
    if (fake::on_kernel() && !fake::stream(s)->capturing) fake::on_kernel()(name, args);
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n)
{
    FAKE("hipMalloc");
    *p = std::calloc(1, n);
    fake::device_memory()[*p] = n;
    ++fake::made_on()[fake::device()];
    return hipSuccess;
}
hipError_t hipFree(void *p) { ++fake::calls()["hipFree"]; fake::device_memory().erase(p); std::free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { FAKE("hipHostMalloc"); *p = std::calloc(1, n); return hipSuccess; }
hipError_t hipHostFree(void *p) { ++fake::calls()["hipHostFree"]; std::free(p); return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { FAKE("hipMemcpy"); std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st)
{
    FAKE("hipMemcpyAsync");
    ++fake::calls()[k == hipMemcpyHostToDevice ? "to device" : k == hipMemcpyDeviceToHost ? "to host" : "on device"];
    std::memcpy(d, s, n);
    ++fake::stream(st)->queued;
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st)
{
    FAKE("hipMemsetAsync");
    std::memset(d, v, n);
    ++fake::stream(st)->queued;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    FAKE("hipStreamCreateWithFlags");
    *s = new ihipStream_t;
    ++fake::made_on()[fake::device()];
    fake::streams().push_back(*s);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s)
{
    auto &v = fake::streams();
    for (size_t k = 0; k < v.size(); ++k) if (v[k] == s) { v.erase(v.begin() + (long)k); break; }
    return hipSuccess;      // (kept: events may name it)
}
hipError_t hipStreamSynchronize(hipStream_t s)
{
    FAKE("hipStreamSynchronize");
    fake::settle(fake::stream(s), fake::stream(s)->queued);
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned)
{
    FAKE("hipStreamWaitEvent");
    if (e->stream && e->stream != fake::stream(s)) fake::stream(s)->waits.push_back({e->stream, e->at});
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { FAKE("hipEventCreate"); *e = new ihipEvent_t; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { FAKE("hipEventCreateWithFlags"); *e = new ihipEvent_t; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    FAKE("hipEventRecord");
    e->stream = fake::stream(s);
    e->at = e->stream->queued;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e)
{
    FAKE("hipEventSynchronize");
    if (e->stream) fake::settle(e->stream, e->at);
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }
hipError_t hipSetDevice(int d) { fake::device() = d; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = fake::device(); return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 2; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    std::memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    p->sharedMemPerBlock = 160 * 1024;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 100000; return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { FAKE("hipFuncSetAttribute"); return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t)
{
    FAKE("hipOccupancyMaxActiveBlocksPerMultiprocessor");
    *n = 1;
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t) { *f = *t = (size_t)64 << 30; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "an error of the check"; }
hipError_t hipGetSymbolAddress(void **p, const void *s) { *p = const_cast<void *>(s); return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode)
{
    FAKE("hipStreamBeginCapture");
    fake::stream(s)->capturing = true;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g)
{
    fake::stream(s)->capturing = false;
    *g = new ihipGraph{1};
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
    FAKE("hipGraphInstantiate");
    *e = new hipGraphExec{1};
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { delete g; return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { delete e; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t s)
{
    FAKE("hipGraphLaunch");
    ++fake::stream(s)->queued;
    if (fake::on_graph()) fake::on_graph()();
    return hipSuccess;
}
}  // extern "C"
