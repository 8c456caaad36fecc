// The HIP runtime calls of libdashinfer_hip.so and libdashinfer_hip_ops.so on host memory, each by its name in a log: what the host
// layer allocates, frees, waits for and launches, and in which order, without a GPU.  Kernels do nothing.  Built and loaded (RTLD_GLOBAL, before
// those libraries) by tests/test_host_runner_cpu.py in a process of its own.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

namespace {
std::mutex mu;
std::vector<std::string> calls;
bool capturing = false;
struct Block { void* p; size_t n; };
std::vector<Block> blocks;
hipError_t note(const char* what) {
  std::lock_guard<std::mutex> g(mu);
  calls.push_back(what);
  return hipSuccess;
}
hipError_t give(void** p, size_t n, const char* what) {
  *p = calloc(1, n ? n : 1);
  std::lock_guard<std::mutex> g(mu);
  blocks.push_back({*p, n});
  calls.push_back(what);
  return hipSuccess;
}
thread_local struct { dim3 g, b; size_t lds; hipStream_t s; } conf;
int handle;
}  // namespace

extern "C" {
void stand_in_clear() { std::lock_guard<std::mutex> g(mu); calls.clear(); }
// the log, one name per line
size_t stand_in_log(char* out, size_t cap) {
  std::lock_guard<std::mutex> g(mu);
  std::string s;
  for (auto& c : calls) s += c + "\n";
  if (out && cap > s.size()) memcpy(out, s.c_str(), s.size() + 1);
  return s.size();
}
// the newest allocation of exactly n bytes
void* stand_in_block(size_t n) {
  std::lock_guard<std::mutex> g(mu);
  for (size_t i = blocks.size(); i-- > 0;)
    if (blocks[i].n == n) return blocks[i].p;
  return nullptr;
}

hipError_t hipMalloc(void** p, size_t n) { return give(p, n, "hipMalloc"); }
hipError_t hipExtMallocWithFlags(void** p, size_t n, unsigned) { return give(p, n, "hipExtMallocWithFlags"); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return give(p, n, "hipHostMalloc"); }
hipError_t hipFree(void*) { return note("hipFree"); }          // (kept: the process is short)
hipError_t hipHostFree(void*) { return note("hipHostFree"); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { memmove(d, s, n); return note("hipMemcpy"); }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { if (!capturing) memmove(d, s, n); return note("hipMemcpyAsync"); }
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, hipMemcpyKind, hipStream_t) {
  for (size_t i = 0; i < h; ++i) memmove((char*)d + i * dp, (const char*)s + i * sp, w);
  return note("hipMemcpy2DAsync");
}
hipError_t hipMemset(void* d, int v, size_t n) { memset(d, v, n); return note("hipMemset"); }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { memset(d, v, n); return note("hipMemsetAsync"); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)&handle; return note("hipEventCreate"); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return note("hipEventRecord"); }
hipError_t hipEventSynchronize(hipEvent_t) { return note("hipEventSynchronize"); }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)&handle; return note("hipStreamCreate"); }
hipError_t hipStreamSynchronize(hipStream_t) { return note("hipStreamSynchronize"); }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return note("hipStreamWaitEvent"); }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* st) { *st = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { capturing = true; return note("hipStreamBeginCapture"); }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { capturing = false; *g = (hipGraph_t)&handle; return note("hipStreamEndCapture"); }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) { *e = (hipGraphExec_t)&handle; return note("hipGraphInstantiate"); }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return note("hipGraphLaunch"); }
hipError_t hipGraphDestroy(hipGraph_t) { return note("hipGraphDestroy"); }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return note("hipGraphExecDestroy"); }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stand-in"; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) { *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 0; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  memset(p, 0, sizeof *p);
  p->multiProcessorCount = 256;
  p->warpSize = 64;
  strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 1; return hipSuccess; }
hipError_t hipIpcCloseMemHandle(void*) { return hipSuccess; }
hipError_t hipIpcGetMemHandle(hipIpcMemHandle_t*, void*) { return hipErrorNotSupported; }
hipError_t hipIpcOpenMemHandle(void**, hipIpcMemHandle_t, unsigned) { return hipErrorNotSupported; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return note(capturing ? "captured launch" : "launch"); }
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) { conf = {g, b, lds, s}; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) { *g = conf.g; *b = conf.b; *lds = conf.lds; *s = conf.s; return hipSuccess; }
void** __hipRegisterFatBinary(const void*) { static void* h[2]; return h; }
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, uint3*, uint3*, dim3*, dim3*, int*) {}
void __hipUnregisterFatBinary(void**) {}
}
