// A HIP runtime of host memory for tests of the library's host side.
//
// Linked with the objects of libskity_hip.so in place of the real runtime, it
// runs no kernel.  It keeps, for every stream, how many kernels were launched
// on it and up to which one the host has waited (through stream and event
// waits, also of other streams), logs the kernels' names, grids and hardware
// queues (streams take them in turn) in launch order, and refuses allocations
// and launches on request, with the error left behind as the real runtime
// leaves it.  The two kernels whose results steer the host, the flatten (bounds
// and edge counts) and the sort (active-edge bounds), write what the test set
// for the frame.  Device time is one millisecond per kernel.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "../../skity_amd/csrc/hipr_common.hpp"

namespace {

typedef std::map<int, int64_t> Clock;  // stream -> launches
struct Stream {
  int id;
  Clock known;  // launches ordered before the stream's end
};
struct Event {
  Clock known;
  double ms;
};
struct Config {
  dim3 grid, block;
  size_t lds;
  hipStream_t stream;
};

// (kernels are registered before this file's other objects are made)
std::map<const void*, std::string>& Names() {
  static std::map<const void*, std::string> names;
  return names;
}
std::vector<Config> g_config;
Clock g_launched, g_done;
int g_streams = 0;
constexpr int kQueues = 4;
double g_ms = 0;
hipError_t g_error = hipSuccess;
std::string g_log;
int64_t g_copied = 0;      // bytes copied from device to device
size_t g_malloc_limit = ~(size_t)0;
std::string g_fail_name;   // the launch of a kernel of this name to refuse
int g_fail_at = -1;

// the frame: per job, modulo their number
std::vector<float> g_ltrb;
std::vector<int32_t> g_edges, g_bound;

void Merge(Clock* into, const Clock& from) {
  for (auto& k : from) (*into)[k.first] = std::max((*into)[k.first], k.second);
}
hipError_t Fail(hipError_t e) { return g_error = e; }

void Flatten(void** args) {
  const int n = *(int*)args[1];
  hipr::JobGeo* geo = *(hipr::JobGeo**)args[7];
  const int32_t* list = *(const int32_t**)args[8];
  for (int i = 0; i < n; i++) {
    const int j = list ? list[i] : i;
    const size_t k = j % g_edges.size();
    hipr::JobGeo g{};
    g.l = g_ltrb[4 * k];
    g.t = g_ltrb[4 * k + 1];
    g.r = g_ltrb[4 * k + 2];
    g.b = g_ltrb[4 * k + 3];
    g.edges = g_edges[k];
    g.cl = g.ct = -hipr::kCullExtent;
    g.cr = g.cb = hipr::kCullExtent;
    geo[j] = g;
  }
}
void Sort(void** args) {
  const int32_t* list = *(const int32_t**)args[0];
  const int n = *(int*)args[1];
  int32_t* bound = *(int32_t**)args[7];
  for (int i = 0; bound && i < n; i++) bound[list[i]] = g_bound[list[i] % g_bound.size()];
}

}  // namespace

#define TEST_API extern "C" __attribute__((visibility("default")))

// ---- what a test sets and asks ---------------------------------------------------
TEST_API void test_set_frame(int n, const float* ltrb, const int32_t* edges,
                             const int32_t* bound) {
  g_ltrb.assign(ltrb, ltrb + 4 * n);
  g_edges.assign(edges, edges + n);
  g_bound.assign(bound, bound + n);
}
TEST_API void test_limit_malloc(int64_t bytes) {
  g_malloc_limit = bytes < 0 ? ~(size_t)0 : (size_t)bytes;
}
// The launch number `at` (from 0 on) of a kernel whose name holds `name`.
TEST_API void test_fail_launch(const char* name, int at) {
  g_fail_name = name;
  g_fail_at = at;
}
TEST_API int64_t test_unfinished() {
  int64_t n = 0;
  for (auto& k : g_launched) n += k.second - g_done[k.first];
  return n;
}
TEST_API int64_t test_copied() { return g_copied; }
TEST_API const char* test_log() { return g_log.c_str(); }
TEST_API void test_reset() {
  g_log.clear();
  g_copied = 0;
  g_fail_at = -1;
  g_malloc_limit = ~(size_t)0;
}

// ---- the runtime ------------------------------------------------------------------
extern "C" {

void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, uint3*,
                           uint3*, dim3*, dim3*, int*) {
  Names()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream) {
  g_config.push_back(Config{grid, block, lds, stream});
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream) {
  const Config c = g_config.back();
  g_config.pop_back();
  *grid = c.grid;
  *block = c.block;
  *lds = c.lds;
  *stream = c.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void** args, size_t,
                           hipStream_t stream) {
  const std::string& name = Names()[f];
  if (g_fail_at >= 0 && name.find(g_fail_name) != std::string::npos && g_fail_at-- == 0)
    return Fail(hipErrorLaunchFailure);
  Stream* s = (Stream*)stream;
  s->known[s->id] = ++g_launched[s->id];
  g_log += name + " " + std::to_string(grid.x) + " " + std::to_string(s->id % kQueues) + "\n";
  g_ms += 1;
  if (name.find("FlattenKernel") != std::string::npos) Flatten(args);
  if (name.find("SortGatherKernel") != std::string::npos) Sort(args);
  return hipSuccess;
}

hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
  *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 160 * 1024;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 8;
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = g_error;
  g_error = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t) { return "refused by the test"; }

hipError_t hipMalloc(void** p, size_t bytes) {
  *p = bytes <= g_malloc_limit ? std::calloc(bytes, 1) : nullptr;
  return *p ? hipSuccess : Fail(hipErrorOutOfMemory);
}
hipError_t hipFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  *p = std::calloc(bytes, 1);
  return *p ? hipSuccess : Fail(hipErrorOutOfMemory);
}
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemcpy(void* to, const void* from, size_t bytes, hipMemcpyKind kind) {
  if (kind == hipMemcpyDeviceToDevice) g_copied += (int64_t)bytes;
  if (kind != hipMemcpyDeviceToDevice || bytes <= (64 << 20)) std::memcpy(to, from, bytes);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* to, const void* from, size_t bytes, hipMemcpyKind kind,
                          hipStream_t) {
  return hipMemcpy(to, from, bytes, kind);
}
hipError_t hipMemsetAsync(void* p, int v, size_t bytes, hipStream_t) {
  std::memset(p, v, bytes);
  return hipSuccess;
}
hipError_t hipMemsetD32Async(hipDeviceptr_t p, int v, size_t n, hipStream_t) {
  std::fill_n((int*)p, n, v);
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void**, const void*) { return Fail(hipErrorInvalidSymbol); }

hipError_t hipStreamCreate(hipStream_t* s) {
  *s = (hipStream_t) new Stream{g_streams++, {}};
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  delete (Stream*)s;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  Merge(&g_done, ((Stream*)s)->known);
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  Merge(&((Stream*)s)->known, ((Event*)e)->known);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = (hipEvent_t) new Event{{}, 0};
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) {
  delete (Event*)e;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  *(Event*)e = Event{((Stream*)s)->known, g_ms};
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  Merge(&g_done, ((Event*)e)->known);
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) {
  *ms = (float)(((Event*)b)->ms - ((Event*)a)->ms);
  return hipSuccess;
}

}  // extern "C"
