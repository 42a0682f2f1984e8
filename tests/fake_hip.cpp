// A HIP runtime for CPU tests of the host code above the kernels: device memory
// is host memory, kernels are not run but logged with the step and the fields
// they would work on, and events read a clock that every launch advances by a
// cost per kernel name.
#include <hip/hip_runtime.h>
#include <sys/mman.h>

#include <cstring>
#include <map>
#include <string>
#include <utility>
#include <vector>

#include "rtm_kernels.h"

namespace {
std::map<const void*, std::string> g_name;          // host stub of a kernel -> its mangled name
std::map<char*, size_t> g_mem;                      // live allocations
std::vector<std::pair<std::string, double>> g_cost; // by part of the name
size_t g_used = 0, g_limit = (size_t)288 << 30;
double g_clock = 0.0;
std::string g_log;
struct Launch { dim3 grid, block; size_t shm; hipStream_t s; };
std::vector<Launch> g_conf;

bool alive(const void* p) {
  auto it = g_mem.upper_bound((char*)p);
  if (it == g_mem.begin()) return false;
  --it;
  return (char*)p < it->first + it->second;
}
struct Line {
  std::string t;
  bool dead = false;
  explicit Line(const char* k) : t(k) {}
  Line& num(const char* n, long long v) { t += std::string(" ") + n + "=" + std::to_string(v); return *this; }
  Line& field(const void* p) { dead = dead || (p && !alive(p)); return *this; }
};
bool has(const std::string& s, const char* k) { return s.find(k) != std::string::npos; }
// "k_interiorILi3E..." -> k_interior, first template number 3, ...
void tmpl(const std::string& s, const char* k, Line& l) {
  size_t at = s.find(std::string(k) + "I");
  for (int i = 0; i < 3 && at != std::string::npos; ++i) {
    at = s.find("Li", at);
    if (at == std::string::npos) break;
    l.num(i == 0 ? "nfd" : i == 1 ? "kind" : "cpt", atoi(s.c_str() + at + 2));
    at += 2;
  }
}
}  // namespace

extern "C" {

const char* fake_log() { return g_log.c_str(); }
void fake_clear() { g_log.clear(); }
void fake_limit(size_t bytes) { g_limit = bytes; }
size_t fake_used() { return g_used; }
void fake_cost(const char* part, double ms) { g_cost.emplace_back(part, ms); }

void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*,
                           dim3*, dim3*, int*) { g_name[host] = name; }
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t n, hipStream_t s) {
  g_conf.push_back({g, b, n, s});
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* n, hipStream_t* s) {
  const Launch l = g_conf.back();
  g_conf.pop_back();
  *g = l.grid; *b = l.block; *n = l.shm; *s = l.s;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** a, size_t, hipStream_t) {
  using namespace rtm;
  const std::string& n = g_name[f];
  double ms = 1.0;
  for (auto& c : g_cost)
    if (has(n, c.first.c_str())) ms = c.second;
  g_clock += ms;
  if (has(n, "k_flag_reset")) **(unsigned**)a[0] = 0xffffffffu;
  Line l("");
  if (has(n, "6k_tileI")) {
    const TileArgs& t = *(TileArgs*)a[0];
    l.t = "k_tile";
    tmpl(n, "k_tile", l);
    l.num("k", t.k).num("nt", t.nt).num("nimg", t.nimg);
    l.field(t.u1).field(t.u0).field(t.u2).field(t.q1).field(t.q0).field(t.q2).field(t.m.fs).field(t.m.r1);
  } else if (has(n, "5k_twoI")) {
    const TwoArgs& t = *(TwoArgs*)a[0];
    l.t = "k_two";
    tmpl(n, "k_two", l);
    l.num("k", t.k).num("nt", t.nt).num("zs", t.zs).num("nimg", t.nimg);
    l.num("u1", (long long)t.u1).num("u0", (long long)t.u0).num("ua", (long long)t.ua).num("ub", (long long)t.ub);
    l.field(t.u1).field(t.u0).field(t.ua).field(t.ub).field(t.cp);
  } else if (has(n, "k_interiorI")) {
    const IntArgs& t = *(IntArgs*)a[0];
    l.t = "k_interior";
    tmpl(n, "k_interior", l);
    l.num("k", t.k).num("nt", t.nt).num("zs", t.zs);
    l.num("u1", (long long)t.u1).num("u0", (long long)t.u0).num("u2", (long long)t.u2);
    l.field(t.u1).field(t.u0).field(t.u2).field(t.uk).field(t.ua).field(t.ub);
  } else if (has(n, "k_frame")  && !has(n, "k_frame_lat")) {
    const FrameArgs& t = *(FrameArgs*)a[0];
    const char* k = has(n, "k_frame_quadI") ? "k_frame_quad" : has(n, "k_frame4I") ? "k_frame4" : "k_frame";
    l.t = k;
    tmpl(n, k, l);
    l.num("k", t.k).num("nt", t.nt);
    l.field(t.u1).field(t.u0).field(t.u2).field(t.m.fs).field(t.m.r1);
    if (has(k, "quad")) l.num("qrows", t.qrows).field(t.cp);
  } else if (has(n, "8k_record")) {
    l.t = "k_record";
    l.num("k", *(int*)a[5]).field(*(void**)a[3]).field(*(void**)a[4]);
  } else if (has(n, "11k_snap_save")) {
    l.t = "k_snap_save";
    l.field(*(void**)a[1]);
  } else {
    l.t = n.substr(0, 40);
  }
  g_log += l.t + (l.dead ? " DEAD\n" : "\n");
  return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t n) {
  *p = nullptr;
  if (g_used + n > g_limit) return hipErrorOutOfMemory;
  void* q = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (q == MAP_FAILED) return hipErrorOutOfMemory;
  g_mem[(char*)q] = n;
  g_used += n;
  *p = q;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  auto it = g_mem.find((char*)p);
  if (it == g_mem.end()) return p ? hipErrorInvalidValue : hipSuccess;
  g_used -= it->second;
  munmap(p, it->second);
  g_mem.erase(it);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) { *f = g_limit - g_used; *t = g_limit; return hipSuccess; }
#undef hipHostMalloc
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = calloc(1, n); return hipSuccess; }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpy2D(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, hipMemcpyKind) {
  for (size_t i = 0; i < h; ++i) memcpy((char*)d + i * dp, (const char*)s + i * sp, w);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t) new double(0.0); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { delete (double*)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { *(double*)e = g_clock; return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) {
  *ms = (float)(*(double*)b - *(double*)a);
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { static char b[1 << 20]; *p = b; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)1; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { *g = (hipGraph_t)1; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  *e = (hipGraphExec_t)1;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

}  // extern "C"
