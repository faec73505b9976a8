// Host stand-in for the HIP runtime and the kernel launches, so that the engine's
// own logic (orders of copies and launches, failures half-way, caches) is tested
// without a GPU: device memory is host memory, streams are names, every call that
// matters for an order is logged, and a chosen call can be made to fail.  A kernel
// does nothing but what the host reads back (thermostat states).
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include "batch.hpp"
#include "engine.hpp"
#include "md.hpp"

using namespace rbmdx;

namespace {
std::string g_log;
std::map<std::string, int> g_fail;  // call name -> calls left before one fails
std::map<char*, size_t> g_live;     // device allocations
int g_count_a = 0;                  // list-A count that an evaluation reports
float g_us = 1.f;                   // what an event pair measures
struct Graph {
  std::vector<std::function<void(hipStream_t)>> ops;  // the launching stream
};
Graph* g_capture = nullptr;

void note(const std::string& s) { g_log += s + "\n"; }

bool fails(const char* name) {
  auto it = g_fail.find(name);
  if (it == g_fail.end() || it->second-- > 0) return false;
  g_fail.erase(it);
  return true;
}

std::string on(hipStream_t s) { return " s" + std::to_string((size_t)s); }

hipError_t launch(const std::string& name, hipStream_t s, std::function<void()> f = [] {}) {
  if (fails(name.c_str())) return hipErrorOutOfMemory;
  auto op = [=](hipStream_t q) {
    note(name + on(q));
    f();
  };
  if (g_capture)
    g_capture->ops.push_back(op);
  else
    op(s);
  return hipSuccess;
}

bool live(const void* p) {
  auto it = g_live.upper_bound((char*)p);
  if (it == g_live.begin()) return false;
  --it;
  return (char*)p < it->first + it->second;
}
}  // namespace

extern "C" {
const char* stub_log() { return g_log.c_str(); }
void stub_clear() { g_log.clear(); }
void stub_fail(const char* name, int after) { g_fail[name] = after; }
void stub_counts(int a) { g_count_a = a; }

hipError_t hipMalloc(void** p, size_t n) {
  if (fails("hipMalloc")) return hipErrorOutOfMemory;
  *p = std::calloc(1, n);
  g_live[(char*)*p] = n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  g_live.erase((char*)p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = std::calloc(1, n);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) {
  *d = h;
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) {
  std::memcpy(d, s, n);
  note(k == hipMemcpyHostToDevice ? "h2d" : "d2h");
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
  std::memset(p, 0, sizeof *p);
  p->multiProcessorCount = 256;
  std::strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
  note("sync");
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  note("sync" + on(s));
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "stub error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = nullptr;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = g_us;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = (hipStream_t)(size_t)99;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  g_capture = new Graph;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  *g = (hipGraph_t)g_capture;
  g_capture = nullptr;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
  if (fails("hipGraphInstantiate")) return hipErrorOutOfMemory;
  *x = (hipGraphExec_t) new Graph(*(Graph*)g);
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
  delete (Graph*)g;
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x) {
  delete (Graph*)x;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t s) {
  if (fails("hipGraphLaunch")) return hipErrorOutOfMemory;
  for (auto& op : ((Graph*)x)->ops) op(s);
  return hipSuccess;
}
}  // extern "C"

namespace rbmdx {
hipError_t noalloc_scratch_init(int) { return hipSuccess; }
void* noalloc_scratch(int) {
  static std::vector<char> buf(kNoAllocScratchBytes);
  return buf.data();
}

template <typename R>
hipError_t launch_force(const Dev<R>& d, const StepArgs<R>&, hipStream_t s) {
  const uint16_t* la = d.list_a;
  Ctrl* c = d.ctrl_host;
  const StepHdr* h = d.hdr_ring;
  return launch("force", s, [=] {
    if (!live(la)) note("force reads freed lists");
    for (int k = 0; k < kSlots; ++k)
      if (h[k].force) {
        note("rebuild");
        const_cast<StepHdr*>(h)[k].force = 0;
      }
    c->max_count_a = g_count_a;
  });
}
template <typename R>
hipError_t launch_build(const Dev<R>& d, const StepArgs<R>&, hipStream_t s) {
  Ctrl* c = d.ctrl;
  return launch("build", s, [=] { c->max_count_a = g_count_a; });
}
template <typename R>
hipError_t launch_skin_build(const Dev<R>&, const StepArgs<R>&, hipStream_t s) {
  return launch("skin_build", s);
}
template <typename R>
hipError_t launch_export(const Dev<R>&, const StepArgs<R>&, int, int, hipStream_t s) {
  return launch("export", s);
}
template <typename R>
hipError_t launch_vjp(const Dev<R>&, const VjpDev<R>&, const StepArgs<R>&, hipStream_t s) {
  return launch("vjp", s);
}
template <typename R>
hipError_t launch_type_params(const TypeParams&, int, const int*, R*, int, R*, hipStream_t s) {
  return launch("type_params", s);
}
template <typename R>
hipError_t md_launch_wrap(const MdArrays<R>&, hipStream_t s) {
  return launch("md_wrap", s);
}
template <typename R>
hipError_t md_launch_second(const MdArrays<R>&, const MdParams&, int, hipStream_t s) {
  return launch("md_second", s);
}
template <typename R>
hipError_t md_launch_apply(const MdArrays<R>&, const MdState* in, MdState* out, hipStream_t s) {
  return launch("md_apply", s, [=] {
    *out = *in;
    out->scale = 1.0;
  });
}
hipError_t md_launch_open(const MdParams&, const MdState* in, MdState* out, int64_t,
                          hipStream_t s) {
  return launch("md_open", s, [=] { *out = *in; });
}
// The state's temperature counts the steps that it has seen.
hipError_t md_launch_thermostat(const MdParams&, const double*, int, const double*,
                                const MdState* in, MdState* out, MdState* open, int setup, int,
                                hipStream_t s) {
  return launch("md_thermostat", s, [=] {
    MdState st = *in;
    st.step = setup ? 0 : st.step + 1;
    st.T = setup ? 0.0 : st.T + 1.0;
    st.scale = 0.5;
    *out = st;
    *open = st;
  });
}
int md_init_parts(int64_t) { return 1; }

#define RBMDX_STUB(R)                                                                         \
  template hipError_t launch_force<R>(const Dev<R>&, const StepArgs<R>&, hipStream_t);        \
  template hipError_t launch_build<R>(const Dev<R>&, const StepArgs<R>&, hipStream_t);        \
  template hipError_t launch_skin_build<R>(const Dev<R>&, const StepArgs<R>&, hipStream_t);   \
  template hipError_t launch_export<R>(const Dev<R>&, const StepArgs<R>&, int, int,           \
                                       hipStream_t);                                          \
  template hipError_t launch_vjp<R>(const Dev<R>&, const VjpDev<R>&, const StepArgs<R>&,      \
                                    hipStream_t);                                             \
  template hipError_t launch_type_params<R>(const TypeParams&, int, const int*, R*, int, R*,  \
                                            hipStream_t);                                     \
  template hipError_t md_launch_wrap<R>(const MdArrays<R>&, hipStream_t);                     \
  template hipError_t md_launch_second<R>(const MdArrays<R>&, const MdParams&, int,           \
                                          hipStream_t);                                       \
  template hipError_t md_launch_apply<R>(const MdArrays<R>&, const MdState*, MdState*,        \
                                         hipStream_t)
RBMDX_STUB(float);
RBMDX_STUB(double);

hipError_t batch_set_epoch(long long*, long long, hipStream_t s) {
  return launch("batch_epoch", s);
}
hipError_t batch_launch(const BatchDev&, const PairConst<float>&, int, int, int, int,
                        const BatchRange&, const BatchTune&, int, hipStream_t s) {
  return launch("batch", s);
}
}  // namespace rbmdx
