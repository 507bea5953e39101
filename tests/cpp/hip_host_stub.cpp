// A HIP runtime on the host for tests of the library's host code without a GPU:
// device memory is host memory, copies are copies, kernels are recorded and do
// nothing, and allocations can be refused.  Loaded with RTLD_GLOBAL ahead of
// libljhip.so, whose HIP calls then arrive here (tests/hip_stub.py).  Time is
// counted in launches, a microsecond each, for the events.
//
// Single-threaded.  stub_* functions read and set its state.
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {

struct Launch {
  std::string name;
  dim3 grid, block;
};

struct State {
  std::map<const void*, std::string> kernels;  // host function -> device name
  std::vector<Launch> launches;
  std::map<void*, size_t> live;  // device allocations
  std::map<std::string, void*> symbols;
  std::map<const void*, std::pair<std::string, size_t>> vars;
  size_t refuse_above = ~size_t(0);  // hipMalloc of more bytes fails
  long fail_in = -1;                 // the hipMalloc after that many fails,
  bool fail_once = false;            // or all from there on
  long mallocs = 0, refused = 0, instantiated = 0, graphs = 0, events = 0;
  dim3 grid, block;
  size_t shared = 0;
  hipStream_t stream = nullptr;
  bool capturing = false;
  long clock = 0, captured = 0;       // launches run, and in the present capture
  std::map<const void*, long> times;  // of events; launches of graphs
  hipError_t last = hipSuccess;
};

State& S()
{
  static State* s = new State;  // kernels register before this library's constructors
  return *s;
}

hipError_t note(hipError_t e)
{
  if (e != hipSuccess) S().last = e;
  return e;
}

// zeroed address space that costs memory only where it is written
void* pages(size_t n)
{
  void* p = mmap(nullptr, n ? n : 1, PROT_READ | PROT_WRITE,
                 MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  return p == MAP_FAILED ? nullptr : p;
}

template <class T>
T handle()
{
  return reinterpret_cast<T>(std::malloc(1));
}

}  // namespace

extern "C" {

// ---- the stub's own interface ----
void stub_refuse_above(size_t bytes) { S().refuse_above = bytes; }
void stub_fail_in(long n, int once)
{
  S().fail_in = n;
  S().fail_once = once != 0;
}
long stub_mallocs() { return S().mallocs; }
long stub_refused() { return S().refused; }
long stub_instantiated() { return S().instantiated; }
long stub_graphs() { return S().graphs; }
long stub_events() { return S().events; }
long stub_live() { return (long)S().live.size(); }
size_t stub_live_bytes()
{
  size_t n = 0;
  for (const auto& a : S().live) n += a.second;
  return n;
}
void stub_clear_launches() { S().launches.clear(); }
long stub_num_launches() { return (long)S().launches.size(); }
const char* stub_launch_name(long k) { return S().launches[k].name.c_str(); }
unsigned stub_launch_grid(long k) { return S().launches[k].grid.x; }

// ---- kernels ----
void** __hipRegisterFatBinary(const void*) { return handle<void**>(); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*,
                           dim3*, dim3*, int*)
{
  S().kernels[f] = name;
}
void __hipRegisterVar(void**, void* var, char* name, char*, int, size_t size, int, int)
{
  S().vars[var] = {name, size};
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t st)
{
  S().grid = g;
  S().block = b;
  S().shared = sh;
  S().stream = st;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* sh, hipStream_t* st)
{
  *g = S().grid;
  *b = S().block;
  *sh = S().shared;
  *st = S().stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t, hipStream_t)
{
  S().launches.push_back({S().kernels[f], g, b});
  ++(S().capturing ? S().captured : S().clock);
  return hipSuccess;
}
hipError_t hipExtLaunchKernel(const void* f, dim3 g, dim3 b, void** a, size_t sh, hipStream_t st,
                              hipEvent_t, hipEvent_t, int)
{
  return hipLaunchKernel(f, g, b, a, sh, st);
}
hipError_t hipGetSymbolAddress(void** p, const void* symbol)
{
  const auto& v = S().vars[symbol];
  void*& at = S().symbols[v.first];
  if (!at) at = pages(v.second);
  *p = at;
  return hipSuccess;
}

// ---- memory ----
hipError_t hipMalloc(void** p, size_t n)
{
  State& s = S();
  ++s.mallocs;
  const bool no = n > s.refuse_above || s.fail_in == 0;
  if (s.fail_in > 0 || s.fail_once) --s.fail_in;
  *p = no ? nullptr : pages(n);
  if (!*p) {
    ++s.refused;
    return note(hipErrorOutOfMemory);
  }
  s.live[*p] = n;
  return hipSuccess;
}
hipError_t hipFree(void* p)
{
  const auto a = S().live.find(p);
  if (p && a == S().live.end()) return note(hipErrorInvalidValue);
  if (p) {
    munmap(p, a->second ? a->second : 1);
    S().live.erase(a);
  }
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
  *p = std::calloc(1, n);
  return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind)
{
  std::memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t)
{
  return hipMemcpy(d, s, n, k);
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t)
{
  std::memset(d, v, n);
  return hipSuccess;
}

// ---- device, streams, events, graphs ----
hipError_t hipGetDevice(int* d)
{
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n)
{
  *n = 1;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int)
{
  *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 0;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int)
{
  std::memset(p, 0, sizeof(*p));
  std::strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "refused by the test"; }
hipError_t hipGetLastError()
{
  const hipError_t e = S().last;
  S().last = hipSuccess;
  return e;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
  *s = handle<hipStream_t>();
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode)
{
  S().capturing = true;
  S().captured = 0;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g)
{
  *g = handle<hipGraph_t>();
  S().times[*g] = S().captured;
  S().capturing = false;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t)
{
  *e = handle<hipGraphExec_t>();
  S().times[*e] = S().times[g];
  ++S().instantiated;
  ++S().graphs;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t)
{
  S().clock += S().times[e];
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t)
{
  --S().graphs;
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e)
{
  *e = handle<hipEvent_t>();
  ++S().events;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t)
{
  --S().events;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t)
{
  S().times[e] = S().clock;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b)
{
  *ms = 1e-3f * (float)(S().times[b] - S().times[a]);
  return hipSuccess;
}

}  // extern "C"
