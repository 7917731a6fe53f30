// A HIP runtime without a GPU, for tests of the library's host code on the
// CPU: loaded RTLD_GLOBAL before libprism_hip.so, whose HIP calls then bind
// here (tests/fake_hip.py).  Device addresses are numbers that nothing is
// stored at; kernels do not run.  It keeps
//  * a log: one line for every allocation, free, wait, destruction, graph
//    launch and kernel launch, in order;
//  * which graph executables may still be running: launched and since then
//    neither their stream nor the device waited for (hipFree waits for the
//    device).  Destroying an executable, a graph, a stream that one runs on or
//    one that was captured on while any runs logs "IN FLIGHT" after the call;
//  * the live device allocations, for checks of the pointers that kernels get.
#define __HIP_PLATFORM_AMD__
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <vector>

namespace {
std::vector<std::string> g_log;
std::map<const void*, std::string> g_names;  // kernels' host functions
std::map<uintptr_t, size_t> g_live;
uintptr_t g_next = (uintptr_t)1 << 44;
uintptr_t g_handle = 0x1000;  // streams, events, graphs
std::map<void*, void*> g_running;  // graph executable -> its last launch's stream
std::set<void*> g_captured;        // streams that a graph was captured on
void* g_capturing = nullptr;       // the caller's stream under capture
size_t g_refuse = (size_t)-1;  // device allocations of this size and more fail
void (*g_on_launch)(const char*, const unsigned*, void**, void*) = nullptr;

void say(const char* what, const void* p) {
  char b[96];
  snprintf(b, sizeof b, "%s %p", what, p);
  g_log.push_back(b);
}
void say_destroy(const char* what, const void* p, bool running = !g_running.empty()) {
  char b[96];
  snprintf(b, sizeof b, "%s %p%s", what, p, running ? " IN FLIGHT" : "");
  g_log.push_back(b);
}
hipError_t give(void** p, size_t n, const char* what) {
  if (n >= g_refuse) return hipErrorOutOfMemory;
  *p = reinterpret_cast<void*>(g_next);
  g_live[g_next] = n;
  g_next += (n + 0xFFFF) / 0x10000 * 0x10000 + 0x10000;
  say(what, *p);
  return hipSuccess;
}
void* handle() { return reinterpret_cast<void*>(g_handle += 16); }
dim3 g_grid, g_block;
size_t g_lds;
hipStream_t g_stream;
}  // namespace

extern "C" {

// ---- what the tests call
size_t fake_log_size() { return g_log.size(); }
const char* fake_log_line(size_t i) { return g_log[i].c_str(); }
void fake_log_clear() { g_log.clear(); }
void fake_on_launch(void (*fn)(const char*, const unsigned*, void**, void*)) { g_on_launch = fn; }
void fake_set_capturing(void* stream) { g_capturing = stream; }
void fake_refuse(size_t bytes) { g_refuse = bytes; }
// bytes from p to the end of the live allocation it lies in, 0 if in none
size_t fake_room(uintptr_t p) {
  auto it = g_live.upper_bound(p);
  if (it == g_live.begin()) return 0;
  --it;
  return p < it->first + it->second ? it->first + it->second - p : 0;
}

// ---- registration and launches
void** __hipRegisterFatBinary(const void*) {
  static void* m;
  return &m;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*,
                           int*) {
  g_names[host] = name;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t st) {
  g_grid = grid, g_block = block, g_lds = lds, g_stream = st;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* st) {
  *grid = g_grid, *block = g_block, *lds = g_lds, *st = g_stream;
  return hipSuccess;
}
const char* hipKernelNameRefByPtr(const void* fn, hipStream_t) {
  auto it = g_names.find(fn);
  return it == g_names.end() ? nullptr : it->second.c_str();
}
hipError_t hipLaunchKernel(const void* fn, dim3 grid, dim3 block, void** args, size_t, hipStream_t st) {
  const char* raw = hipKernelNameRefByPtr(fn, st);
  int rc = 0;
  char* dem = raw ? abi::__cxa_demangle(raw, nullptr, nullptr, &rc) : nullptr;
  const std::string name = dem ? dem : raw ? raw : "?";
  free(dem);
  g_log.push_back("launch " + name);
  const unsigned dims[6] = {grid.x, grid.y, grid.z, block.x, block.y, block.z};
  if (g_on_launch) g_on_launch(name.c_str(), dims, args, st);
  return hipSuccess;
}

// ---- device
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950:sramecc+:xnack-");
  p->multiProcessorCount = 256;
  p->sharedMemPerBlock = 160 << 10;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
  g_log.push_back("device wait");
  g_running.clear();
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error of the fake runtime"; }

// ---- memory
hipError_t hipMalloc(void** p, size_t n) { return give(p, n, "malloc"); }
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t) { return give(p, n, "malloc async"); }
hipError_t hipMallocFromPoolAsync(void** p, size_t n, hipMemPool_t, hipStream_t) { return give(p, n, "malloc pool"); }
hipError_t hipFree(void* p) {
  g_running.clear();  // waits for the device
  g_live.erase(reinterpret_cast<uintptr_t>(p));
  say("free", p);
  return hipSuccess;
}
hipError_t hipFreeAsync(void* p, hipStream_t) {
  g_live.erase(reinterpret_cast<uintptr_t>(p));
  say("free async", p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return (*p = malloc(n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void* p) { return free(p), hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { return *d = h, hipSuccess; }
hipError_t hipMemcpy(void*, const void*, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipMemPoolCreate(hipMemPool_t* p, const hipMemPoolProps*) {
  return *p = static_cast<hipMemPool_t>(handle()), hipSuccess;
}
hipError_t hipMemPoolDestroy(hipMemPool_t) { return hipSuccess; }
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void*) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static void* scratch;
  if (!scratch && give(&scratch, (size_t)64 << 20, "symbol") != hipSuccess) return hipErrorOutOfMemory;
  return *p = scratch, hipSuccess;
}

// ---- streams, events, graphs
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  return *s = static_cast<hipStream_t>(handle()), hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  bool running = g_captured.count(s) && !g_running.empty();
  for (const auto& r : g_running) running = running || r.second == s;
  return say_destroy("stream destroy", s, running), hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  say("stream wait", s);
  for (auto it = g_running.begin(); it != g_running.end();)
    it = it->second == s ? g_running.erase(it) : ++it;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) { return g_captured.insert(s), hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return *g = static_cast<hipGraph_t>(handle()), hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
  *st = s && s == g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  return *e = static_cast<hipGraphExec_t>(handle()), hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s) {
  say("graph launch", e);
  g_running[e] = s;
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { return say_destroy("exec destroy", e), hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { return say_destroy("graph destroy", g), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = static_cast<hipEvent_t>(handle()), hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }

}  // extern "C"
