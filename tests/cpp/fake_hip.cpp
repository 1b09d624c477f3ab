// fake_hip.cpp - a HIP runtime without a GPU, for tests of the library's host
// side: which kernels a call launches, in which order, with how much LDS, and
// what it does when an allocation fails.  Device memory is host memory, copies
// happen at once, kernels are written down and not run, a captured graph is
// the list of its kernels.  Like the device, it refuses a launch whose LDS is
// above 64 KiB and above what hipFuncSetAttribute allowed its kernel.
#include <hip/hip_runtime_api.h>

#include <cxxabi.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <vector>

namespace {
struct Launch {
  std::string name;
  unsigned grid, block;
  size_t lds;
};
struct Graph {
  std::vector<Launch> launches;
};
struct Call {
  dim3 grid, block;
  size_t lds;
  hipStream_t stream;
};
std::map<const void *, int> lds_limit;
std::vector<std::string> attributes;   // "name bytes", in call order
std::vector<Launch> launches;
std::vector<Call> pushed;
std::set<void *> live;
Graph *capture = nullptr;
long fail_in = -1;      // allocations until one fails, -1: never
long fail_count = 0;    // how many fail from there
hipError_t last = hipSuccess;
std::string text;

// filled by constructors of the library's objects, perhaps before this file's
std::map<const void *, std::string> &names() {
  static std::map<const void *, std::string> m;
  return m;
}
hipError_t err(hipError_t e) {
  if (e != hipSuccess) last = e;
  return e;
}
// "k_pair<512, false>" of a mangled name
std::string demangled(const char *m) {
  int rc = 0;
  char *d = abi::__cxa_demangle(m, nullptr, nullptr, &rc);
  std::string s = rc == 0 ? d : m;
  std::free(d);
  const std::string anon = "(anonymous namespace)::";
  for (size_t p = s.find(anon); p != std::string::npos; p = s.find(anon)) s.erase(p, anon.size());
  s = s.substr(0, s.find('('));
  return s.compare(0, 5, "void ") == 0 ? s.substr(5) : s;
}
hipError_t launch(const void *fn, dim3 g, dim3 b, size_t lds) {
  const auto n = names().find(fn);
  if (n == names().end() || g.x == 0 || g.y != 1 || g.z != 1 || b.x == 0 || b.x > 1024) return err(hipErrorInvalidValue);
  const auto limit = lds_limit.find(fn);
  if (lds > 64 * 1024 && (limit == lds_limit.end() || lds > (size_t)limit->second)) return err(hipErrorInvalidValue);
  (capture ? capture->launches : launches).push_back({n->second, g.x, b.x, lds});
  return hipSuccess;
}
}  // namespace

extern "C" {

// the tests' side
void fake_fail(long in, long count) {
  fail_in = in;
  fail_count = count;
}
const char *fake_launches(int forget) {
  text.clear();
  for (const Launch &l : launches)
    text += l.name + "|" + std::to_string(l.grid) + "|" + std::to_string(l.block) + "|" + std::to_string(l.lds) + "\n";
  if (forget) launches.clear();
  return text.c_str();
}
const char *fake_attributes() {
  text.clear();
  for (const std::string &s : attributes) text += s + "\n";
  return text.c_str();
}
long fake_live() { return (long)live.size(); }

// the runtime's side
void **__hipRegisterFatBinary(const void *) {
  static void *m = nullptr;
  return &m;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *device, unsigned, void *, void *, void *,
                           void *, int *) {
  names()[host] = demangled(device);
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
  pushed.push_back({g, b, lds, s});
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
  *g = pushed.back().grid;
  *b = pushed.back().block;
  *lds = pushed.back().lds;
  *s = pushed.back().stream;
  pushed.pop_back();
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *fn, dim3 g, dim3 b, void **, size_t lds, hipStream_t) {
  return launch(fn, g, b, lds);
}
hipError_t hipLaunchCooperativeKernel(const void *fn, dim3 g, dim3 b, void **, unsigned lds, hipStream_t) {
  return launch(fn, g, b, lds);
}
hipError_t hipFuncSetAttribute(const void *fn, hipFuncAttribute a, int v) {
  if (a == hipFuncAttributeMaxDynamicSharedMemorySize) {
    lds_limit[fn] = v;
    attributes.push_back(names()[fn] + "|" + std::to_string(v));
  }
  return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) {
  if (fail_in == 0 && fail_count > 0) {
    --fail_count;
    *p = nullptr;
    return err(hipErrorOutOfMemory);
  }
  if (fail_in > 0) --fail_in;
  *p = std::calloc(1, n ? n : 1);
  live.insert(*p);
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  if (!p) return hipSuccess;
  if (live.erase(p) != 1) std::abort();   // freed twice, or never allocated
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  if (!d || !s) return err(hipErrorInvalidValue);
  if (!capture) std::memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
  if (!d) return err(hipErrorInvalidValue);
  if (!capture) std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t) {
  *f = *t = (size_t)256 << 30;
  return hipSuccess;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t *, size_t *, hipDeviceptr_t) { return err(hipErrorInvalidValue); }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) { return err(hipErrorInvalidValue); }
hipError_t hipGetSymbolAddress(void **p, const void *) {
  static char symbol;   // an address is all that the tests ask of it
  *p = &symbol;
  return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
  *v = 256;   // the only one asked for: compute units
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t) { return "fake runtime"; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(std::malloc(1));
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  std::free(s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  capture = new Graph;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
  *g = reinterpret_cast<hipGraph_t>(capture);
  capture = nullptr;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t g, hipGraphNode_t *, char *, size_t) {
  *x = reinterpret_cast<hipGraphExec_t>(new Graph(*reinterpret_cast<Graph *>(g)));
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t) {
  const auto &l = reinterpret_cast<Graph *>(x)->launches;
  launches.insert(launches.end(), l.begin(), l.end());
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
  delete reinterpret_cast<Graph *>(g);
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x) {
  delete reinterpret_cast<Graph *>(x);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  std::free(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = 1.0f;
  return hipSuccess;
}

}  // extern "C"
