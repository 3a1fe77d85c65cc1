/*
 * device_stub.cpp -- a stand-in for the HIP runtime that runs the library's
 * host code without a GPU: device memory is host memory, copies are
 * copies, kernels do nothing.  Loaded with global symbols before the
 * library, so the library's runtime calls come here.
 *
 * It counts launches by kernel name and allocations, lets the n-th
 * allocation from now fail, and checks what a launch would have read: every
 * pointer among a kernel's arguments must be null or lie in an allocation
 * that is still there (in a captured graph, at the time of its launch) and
 * on the device that is current, and the pointers of two-step passes and of the network's forward kernels must
 * not be null.  Freed memory stays reserved, so a stale pointer is never
 * taken for a new one.
 */
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>

#include <cxxabi.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <string>
#include <vector>

#include "cs_pass2.h"

#undef hipGetDeviceProperties

namespace {

struct Block {
  size_t bytes;
  bool live;
  int device;
};
int g_device = 0;
std::map<uintptr_t, Block> g_blocks;   /* by first byte */
std::map<const void*, std::string> g_names;
std::map<std::string, long> g_launches;
std::vector<std::string> g_bad;
hipError_t g_last = hipSuccess;
long g_allocs = 0, g_fail_in = -1;

struct Launch {
  std::string name;
  std::vector<const void*> ptrs;
  bool need_all;
};
std::vector<Launch>* g_capture = nullptr;

hipError_t fail(hipError_t e) { return g_last = e; }

/* 1: in a live allocation of the current device, 2: of another, 0: in none,
 * -1: in a freed one */
int where(const void* p)
{
  auto it = g_blocks.upper_bound((uintptr_t)p);
  if (it == g_blocks.begin()) return 0;
  --it;
  if ((uintptr_t)p >= it->first + it->second.bytes) return 0;
  return !it->second.live ? -1 : it->second.device == g_device ? 1 : 2;
}

void check(const Launch& l)
{
  g_launches[l.name]++;
  for (size_t k = 0; k < l.ptrs.size(); k++) {
    const void* p = l.ptrs[k];
    if (p ? where(p) == 1 : !l.need_all) continue;
    char msg[64];
    const int at = p ? where(p) : 0;
    snprintf(msg, sizeof msg, ": pointer %zu is %s", k,
             !p ? "null" : at == 2 ? "on another device" : at ? "freed" : "no device memory");
    g_bad.push_back(l.name + msg);
  }
}

/* The parameter types of a demangled kernel, at the outermost commas. */
std::vector<std::string> params(const std::string& sig)
{
  std::vector<std::string> out;
  const size_t end = sig.rfind(')');
  if (end == std::string::npos) return out;
  int depth = 0;
  size_t begin = end;
  while (begin-- > 0) {
    if (sig[begin] == ')' || sig[begin] == '>') depth++;
    if (sig[begin] == '<') depth--;
    if (sig[begin] == '(' && depth-- == 0) break;
  }
  std::string cur;
  depth = 0;
  for (size_t k = begin + 1; k < end; k++) {
    const char ch = sig[k];
    if (ch == '<' || ch == '(') depth++;
    if (ch == '>' || ch == ')') depth--;
    if (ch == ',' && depth == 0) {
      out.push_back(cur);
      cur.clear();
    } else {
      cur += ch;
    }
  }
  if (!cur.empty()) out.push_back(cur);
  return out;
}

/* Streams and events are only names. */
char g_handle[1 << 16];
size_t g_handles = 0;
template <typename H>
hipError_t handle(H* h)
{
  *h = (H)(g_handle + g_handles++ % sizeof g_handle);
  return hipSuccess;
}

}  // namespace

extern "C" {

/* ------------------------------------------------ what the tests use */

void stub_fail_alloc_in(long n) { g_fail_in = n; }   /* 0: the next one, -1: none */
long stub_allocs(void) { return g_allocs; }
long stub_live_bytes(void)
{
  long n = 0;
  for (const auto& kv : g_blocks)
    if (kv.second.live) n += (long)kv.second.bytes;
  return n;
}
long stub_launches(const char* part)
{
  long n = 0;
  for (const auto& kv : g_launches)
    if (kv.first.find(part) != std::string::npos) n += kv.second;
  return n;
}
long stub_bad(void) { return (long)g_bad.size(); }
const char* stub_bad_at(long k) { return g_bad[(size_t)k].c_str(); }
int stub_pending_error(void) { return (int)g_last; }
int stub_zlimit(uint64_t group, uint64_t nz, uint64_t pad) { return p2_zlimit(group, nz, pad); }

/* ------------------------------------------------------- the runtime */

void** __hipRegisterFatBinary(const void*)
{
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* device, unsigned, void*, void*, void*, void*,
                           int*)
{
  int st = 0;
  std::unique_ptr<char, void (*)(void*)> d(abi::__cxa_demangle(device, nullptr, nullptr, &st), free);
  g_names[host] = st == 0 ? d.get() : device;
}
static std::map<const void*, void*> g_vars;
void __hipRegisterVar(void**, void* var, char*, char*, int, size_t size, int, int)
{
  void* p = calloc(1, size);
  g_blocks[(uintptr_t)p] = Block{size, true, 0};
  g_vars[var] = p;
}
static struct { dim3 grid, block; size_t shmem; hipStream_t stream; } g_config;
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, hipStream_t stream)
{
  g_config = {grid, block, shmem, stream};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shmem, hipStream_t* stream)
{
  *grid = g_config.grid;
  *block = g_config.block;
  *shmem = g_config.shmem;
  *stream = g_config.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t, hipStream_t)
{
  Launch l{g_names[f], {}, false};
  if (!grid.x || !grid.y || !grid.z || !block.x) {
    g_bad.push_back(l.name + ": empty grid");
    return fail(hipErrorInvalidConfiguration);
  }
  const std::vector<std::string> ts = params(l.name);
  for (size_t k = 0; k < ts.size(); k++)
    if (ts[k].find('*') != std::string::npos) l.ptrs.push_back(*(void* const*)args[k]);
  if (l.name.find("k_pass2") != std::string::npos) {
    const P2Args& a = *(const P2Args*)args[0];
    l.need_all = true;
    l.ptrs = {a.u, a.un, a.words, a.params, a.geos, a.tiles, a.col_start, a.vz, a.fsum, a.l1};
  }
  l.need_all = l.need_all || l.name.find("k_mlp_to_bf16") != std::string::npos ||
               l.name.find("k_mlp_forward") != std::string::npos;
  if (g_capture) g_capture->push_back(l);
  else check(l);
  return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t bytes)
{
  g_allocs++;
  if (g_fail_in >= 0 && g_fail_in-- == 0) return fail(hipErrorOutOfMemory);
  *p = calloc(1, bytes ? bytes : 1);
  g_blocks[(uintptr_t)*p] = Block{bytes, true, g_device};
  return hipSuccess;
}
hipError_t hipFree(void* p)
{
  if (!p) return hipSuccess;
  auto it = g_blocks.find((uintptr_t)p);
  if (it == g_blocks.end() || !it->second.live) {
    g_bad.push_back("hipFree of what is not allocated");
    return fail(hipErrorInvalidValue);
  }
  it->second.live = false;
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned)
{
  *p = calloc(1, bytes);
  return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
  free(p);
  return hipSuccess;
}
static hipError_t copy(void* dst, const void* src, size_t bytes, hipMemcpyKind kind)
{
  auto outside = [bytes](const void* p) { return bytes && (where(p) != 1 || where((const char*)p + bytes - 1) != 1); };
  if ((kind != hipMemcpyDeviceToHost && outside(dst)) || (kind != hipMemcpyHostToDevice && outside(src))) {
    g_bad.push_back("a copy outside device memory");
    return fail(hipErrorInvalidValue);
  }
  memmove(dst, src, bytes);
  return hipSuccess;
}
hipError_t hipMemcpy(void* dst, const void* src, size_t bytes, hipMemcpyKind kind) { return copy(dst, src, bytes, kind); }
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, hipStream_t)
{
  return copy(dst, src, bytes, kind);
}
hipError_t hipMemcpy2DAsync(void* dst, size_t dpitch, const void* src, size_t spitch, size_t width, size_t height,
                            hipMemcpyKind kind, hipStream_t)
{
  for (size_t k = 0; k < height; k++) {
    const hipError_t e = copy((char*)dst + k * dpitch, (const char*)src + k * spitch, width, kind);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* dst, int value, size_t bytes, hipStream_t)
{
  if (bytes && (where(dst) != 1 || where((char*)dst + bytes - 1) != 1)) {
    g_bad.push_back("a fill outside device memory");
    return fail(hipErrorInvalidValue);
  }
  memset(dst, value, bytes);
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* var)
{
  *p = g_vars[var];
  return hipSuccess;
}

hipError_t hipGetDevice(int* d)
{
  *d = g_device;
  return hipSuccess;
}
hipError_t hipSetDevice(int d)
{
  g_device = d;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int)
{
  memset(p, 0, sizeof *p);
  strcpy(p->name, "stand-in");
  strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetLastError(void)
{
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "an error"; }

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return handle(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return handle(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return handle(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t)
{
  *ms = 1.0f;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode)
{
  g_capture = new std::vector<Launch>();
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g)
{
  *g = (hipGraph_t)g_capture;
  g_capture = nullptr;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t g, hipGraphNode_t*, char*, size_t)
{
  *x = (hipGraphExec_t) new std::vector<Launch>(*(std::vector<Launch>*)g);
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t)
{
  for (const Launch& l : *(std::vector<Launch>*)x) check(l);
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x)
{
  delete (std::vector<Launch>*)x;
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g)
{
  delete (std::vector<Launch>*)g;
  return hipSuccess;
}

}  // extern "C"
