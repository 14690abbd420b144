// Host stand-in for the HIP runtime calls of libhelios_ccsd, so that a test
// without a device can follow what the library's host code asks for: device
// memory is host memory, a launch is written down (kernel, grid, and which of
// its pointer arguments are null) and runs nothing, except that the first
// stub_running() molecules stay active in a solve, and an allocation can be made
// to fail.  Loaded with RTLD_GLOBAL before the library, whose undefined
// runtime symbols then resolve here first.
#include <cxxabi.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
struct Dim3 {
  unsigned x, y, z;
};
struct Kernel {
  std::string name;
  std::vector<bool> pointer;   // per parameter
};
std::map<const void*, Kernel> kernels;
std::map<void*, size_t> blocks;
size_t held = 0, peak = 0;
long allocations = 0, fail_at = 0;
int running = 0;   // molecules that a solve's reset kernel leaves active
std::string launches;
thread_local Dim3 call_grid, call_block;
thread_local size_t call_shared;
thread_local void* call_stream;

// "void ns::k<..>(A*, B const*, int)" -> name and which parameters are pointers
Kernel parse(const char* mangled) {
  int status = 0;
  char* text = abi::__cxa_demangle(mangled, nullptr, nullptr, &status);
  Kernel k;
  k.name = status == 0 ? text : mangled;
  free(text);
  if (k.name.empty() || k.name.back() != ')') return k;
  size_t open = k.name.size() - 1;
  for (int depth = 0;; --open) {
    depth += k.name[open] == ')' ? 1 : (k.name[open] == '(' ? -1 : 0);
    if (depth == 0 || open == 0) break;
  }
  const std::string args = k.name.substr(open + 1, k.name.size() - open - 2);
  int depth = 0;
  char last = 0;
  for (char c : args + ",") {
    if (c == ',' && depth == 0) {
      k.pointer.push_back(last == '*');
      last = 0;
      continue;
    }
    depth += c == '<' || c == '(' ? 1 : (c == '>' || c == ')' ? -1 : 0);
    if (c != ' ') last = c;
  }
  k.name.resize(open);
  return k;
}
}  // namespace

extern "C" {
// test controls: the n-th allocation from now fails (0: none)
void stub_fail_at(long n) { fail_at = n; }
long stub_allocations() { return allocations; }
void stub_running(int n) { running = n; }
size_t stub_held() { return held; }
size_t stub_peak(int reset) {
  if (reset) peak = held;
  return peak;
}
const char* stub_launches() { return launches.c_str(); }
void stub_clear() { launches.clear(); }

void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* device, unsigned, void*, void*, void*, void*, int*) {
  kernels[host] = parse(device);
}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shared, void* stream) {
  call_grid = grid, call_block = block, call_shared = shared, call_stream = stream;
  return 0;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* shared, void** stream) {
  *grid = call_grid, *block = call_block, *shared = call_shared, *stream = call_stream;
  return 0;
}
int hipLaunchKernel(const void* host, Dim3 grid, Dim3 block, void** args, size_t, void*) {
  const Kernel& k = kernels[host];
  launches += k.name + " " + std::to_string(grid.x) + "x" + std::to_string(block.x) + " ";
  for (size_t q = 0; q < k.pointer.size(); ++q)
    if (k.pointer[q]) launches += *static_cast<void**>(args[q]) == nullptr ? '0' : '1';
  launches += '\n';
  if (k.name.find("k_reset_state") != std::string::npos) {   // (State*, int* active, int molecules)
    int* const active = *static_cast<int**>(args[1]);
    for (int q = 0, n = *static_cast<int*>(args[2]); q < n; ++q) active[q] = q < running;
  }
  return 0;
}

int hipMalloc(void** p, size_t bytes) {
  ++allocations;
  *p = nullptr;
  if (fail_at > 0 && --fail_at == 0) return 2;   // hipErrorOutOfMemory
  *p = calloc(1, bytes ? bytes : 1);
  if (*p == nullptr) return 2;
  blocks[*p] = bytes;
  held += bytes;
  if (held > peak) peak = held;
  return 0;
}
int hipFree(void* p) {
  if (p == nullptr) return 0;
  auto it = blocks.find(p);
  if (it == blocks.end()) abort();   // freed twice or never allocated
  held -= it->second;
  blocks.erase(it);
  free(p);
  return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int) {
  if (n && (d == nullptr || s == nullptr)) return 1;
  memcpy(d, s, n);
  return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void*) { return hipMemcpy(d, s, n, kind); }
int hipMemset(void* d, int v, size_t n) {
  if (n && d == nullptr) return 1;
  memset(d, v, n);
  return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void*) { return hipMemset(d, v, n); }

int hipSetDevice(int) { return 0; }
int hipDeviceGetAttribute(int* v, int, int) {
  *v = 160 * 1024;
  return 0;
}
int hipFuncSetAttribute(const void*, int, int) { return 0; }
int hipDeviceSynchronize() { return 0; }
int hipGetLastError() { return 0; }
const char* hipGetErrorString(int) { return "stub error"; }
int hipStreamCreateWithFlags(void** s, unsigned) {
  *s = malloc(1);
  return 0;
}
int hipStreamDestroy(void* s) {
  free(s);
  return 0;
}
int hipStreamSynchronize(void*) { return 0; }
int hipStreamBeginCapture(void*, int) { return 0; }
int hipStreamEndCapture(void*, void** g) {
  *g = malloc(1);
  return 0;
}
int hipGraphInstantiate(void** e, void*, void*, char*, size_t) {
  *e = malloc(1);
  return 0;
}
int hipGraphLaunch(void*, void*) { return 0; }
int hipGraphDestroy(void* g) {
  free(g);
  return 0;
}
int hipGraphExecDestroy(void* e) {
  free(e);
  return 0;
}
int hipEventCreate(void** e) {
  *e = malloc(1);
  return 0;
}
int hipEventDestroy(void* e) {
  free(e);
  return 0;
}
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*) {
  *ms = 0.f;
  return 0;
}
}
