// A stand-in for the HIP runtime on machines without a GPU, for tests of libt0mi's host side: which kernels
// a call launches, on what grid, and what it does when memory runs out, during capture and with live
// graphs.  Loaded with RTLD_GLOBAL before libt0mi.so, so that its definitions come first.  Nothing is
// executed: device memory is addresses, a launch is a line of text.
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>
#include <string.h>

#include <map>
#include <string>

namespace {
std::map<const void*, std::string> g_names;
std::string g_launches, g_last_name;
hipError_t g_last = hipSuccess;
size_t g_limit = ~(size_t)0, g_allocated = 0;
std::map<uintptr_t, size_t> g_live;
uintptr_t g_next = 0x100000000000ull;
bool g_capturing = false;
size_t g_captured = 0;
dim3 g_grid, g_block;

// hipGetLastError returns the last error of any call, also after calls that succeeded.
hipError_t ret(hipError_t e) {
  if (e != hipSuccess && e != hipErrorNotReady) g_last = e;
  return e;
}
}  // namespace

extern "C" {
// Launches since the last call, one a line: "name grid.x grid.y grid.z block.x".
const char* fake_launches() {
  static std::string out;
  out.swap(g_launches);
  g_launches.clear();
  return out.c_str();
}
// hipMalloc calls above `bytes` fail from now on.
void fake_set_malloc_limit(size_t bytes) { g_limit = bytes; }
size_t fake_allocated() { return g_allocated; }

void** __hipRegisterFatBinary(const void*) {
  static void* h = nullptr;
  return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, dim3*, dim3*,
                           int*) {
  int st = 0;
  char* d = abi::__cxa_demangle(name, nullptr, nullptr, &st);
  g_names[host] = d ? d : name;
  free(d);
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t, hipStream_t) {
  g_grid = grid;
  g_block = block;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shmem, hipStream_t* s) {
  *grid = g_grid;
  *block = g_block;
  *shmem = 0;
  *s = nullptr;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void**, size_t, hipStream_t) {
  auto it = g_names.find(f);
  g_last_name = it == g_names.end() ? "?" : it->second;
  std::string n = g_last_name;
  if (n.rfind("void ", 0) == 0) n = n.substr(5);
  n = n.substr(0, n.rfind('('));  // without the parameters
  for (size_t i; (i = n.find("t0mi::")) != std::string::npos;) n.erase(i, 6);
  std::string flat;
  for (char c : n)
    if (c != ' ') flat += c;
  g_launches += flat + " " + std::to_string(grid.x) + " " + std::to_string(grid.y) + " " + std::to_string(grid.z) + " " +
                std::to_string(block.x) + "\n";
  g_captured += g_capturing;
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
  *p = nullptr;
  if (g_capturing) return ret(hipErrorStreamCaptureUnsupported);
  if (n > g_limit) return ret(hipErrorOutOfMemory);
  *p = (void*)g_next;
  g_live[g_next] = n;
  g_allocated += n;
  g_next += (n + 0xFFFFF) & ~(size_t)0xFFFFF;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (!p) return hipSuccess;
  auto it = g_live.find((uintptr_t)p);
  if (it == g_live.end()) return ret(hipErrorInvalidValue);
  g_allocated -= it->second;
  g_live.erase(it);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void*, size_t n, hipMemcpyKind k, hipStream_t) {
  if (k != hipMemcpyDeviceToHost) return hipSuccess;
  memset(dst, 0, n);
  if (g_last_name.find("placement") != std::string::npos)  // workgroup i on XCD i % 8
    for (size_t i = 0; i < n / 4; ++i) ((uint32_t*)dst)[i] = (uint32_t)(i % 8);
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t e) {
  return e == hipSuccess ? "no error" : e == hipErrorOutOfMemory ? "out of memory" : "error";
}
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {  // hipGetDevicePropertiesR0600 by the header
  memset((void*)p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950:sramecc+:xnack-");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) {
  *p = (void*)0x200000000000ull;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = (hipStream_t)(uintptr_t)0x1000;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return ret(g_capturing ? hipErrorStreamCaptureUnsupported : hipSuccess); }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* st) {
  *st = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  g_capturing = true;
  g_captured = 0;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  g_capturing = false;
  *g = (hipGraph_t)(uintptr_t)0x2000;
  return hipSuccess;
}
hipError_t hipGraphGetNodes(hipGraph_t, hipGraphNode_t*, size_t* n) {
  *n = g_captured;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  *e = (hipGraphExec_t)(uintptr_t)0x3000;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = (hipEvent_t)(uintptr_t)0x4000;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 1.0f;
  return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
}
