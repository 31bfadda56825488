// A HIP runtime of the host alone, for tests of the library's host side where
// no GPU is: memory is host memory, kernels are listed and not run (but for
// the descriptor's upload, whose destination is kept up to date), launches can
// be made to fail and a stream to look like one being captured. Loaded before
// the library with its symbols global, so that the library binds to it.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

#include "../profess_amd/csrc/ofd_internal.h"

namespace {
std::map<const void*, std::string> names;
std::string listed, failing;
hipError_t last = hipSuccess;
bool capturing = false;
int lds = 163840, timings = 0, fastest = 0;
std::map<std::string, unsigned> grids;   // blocks along x of a kernel's last launch
unsigned host_flags = 0;
const ofd::ReqDesc* desc = nullptr;   // the last uploaded or evaluated
struct Call {
  dim3 g, b;
  size_t s;
  hipStream_t st;
} call;
template <typename T> hipError_t give(T** p, size_t n) {
  *p = static_cast<T*>(std::calloc(n, 1));
  return hipSuccess;
}
hipError_t handle(void** p) { return give(p, 16); }
}  // namespace

#define API extern "C" __attribute__((visibility("default")))
API void stub_fail(const char* kernel) { failing = kernel; }
API void stub_capture(int on) { capturing = on != 0; }
API void stub_lds(int bytes) { lds = bytes; }
API void stub_clear() { listed.clear(); }
// the k-th timing from now is half the others
API void stub_fastest(int k) { timings = 0; fastest = k; }
API int stub_grid(const char* kernel) {
  for (const auto& g : grids)
    if (g.first.find(kernel) != std::string::npos) return g.second;
  return 0;
}
API const char* stub_listed() { return listed.c_str(); }
API unsigned stub_host_flags() { return host_flags; }
// fields of the descriptor the last evaluation pass was given
API const ofd::ReqDesc* stub_desc() { return desc; }
API int stub_sizes(int k) { return k == 0 ? sizeof(ofd::ReqDesc) : sizeof(ofd::ShapePlan); }
API const void* stub_u() { return desc->u; }
API const void* stub_out() { return desc->out; }
API const void* stub_u2() { return desc->u2; }
API const void* stub_out2() { return desc->out2; }

API void** __hipRegisterFatBinary(const void*) { return static_cast<void**>(std::calloc(1, 8)); }
API void __hipUnregisterFatBinary(void**) {}
API void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, dim3*, dim3*,
                               int*) {
  names[host] = name;
}
API void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
API hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st) {
  call = {g, b, s, st};
  return hipSuccess;
}
API hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st) {
  *g = call.g; *b = call.b; *s = call.s; *st = call.st;
  return hipSuccess;
}
API hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void** args, size_t, hipStream_t) {
  const std::string& n = names[f];
  if (!failing.empty() && n.find(failing) != std::string::npos) return last = hipErrorLaunchFailure;
  listed += n + "\n";
  grids[n] = grid.x;
  if (n.find("k_put_desc") != std::string::npos) {
    if (!capturing) std::memcpy(*static_cast<void**>(args[1]), args[0], sizeof(ofd::ReqDesc));
    desc = *static_cast<ofd::ReqDesc**>(args[1]);
  } else if (n.find("k_fin") != std::string::npos) {   // also k_finalize: the end of an evaluation
    desc = *static_cast<ofd::ReqDesc**>(args[0]);
  }
  return hipSuccess;
}
API hipError_t hipGetLastError() { const hipError_t e = last; last = hipSuccess; return e; }
API const char* hipGetErrorString(hipError_t) { return "stub"; }
API hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
API hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
API hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = lds; return hipSuccess; }
API hipError_t hipMalloc(void** p, size_t n) { return give(p, n); }
API hipError_t hipFree(void* p) { std::free(p); return hipSuccess; }
API hipError_t hipHostMalloc(void** p, size_t n, unsigned flags) { host_flags = flags; return give(p, n); }
API hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
API hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  if (failing == "hipMemcpyAsync") return hipErrorUnknown;
  std::memcpy(d, s, n);
  return hipSuccess;
}
API hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { std::memset(d, v, n); return hipSuccess; }
API hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
API hipError_t hipGetSymbolAddress(void** p, const void*) { return give(p, 64 << 20); }
API hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return handle((void**)s); }
API hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
API hipError_t hipStreamSynchronize(hipStream_t) { return capturing ? hipErrorStreamCaptureUnsupported : hipSuccess; }
API hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* c) {
  *c = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
API hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
API hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipErrorNotSupported; }
API hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) { return hipErrorNotSupported; }
API hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
API hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
API hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
API hipError_t hipEventCreate(hipEvent_t* e) { return handle((void**)e); }
API hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return handle((void**)e); }
API hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
API hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
API hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
API hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
API hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = ++timings == fastest ? 0.5f : 1.f;
  return hipSuccess;
}
