// The HIP runtime calls of libsgpp_hip.so on host memory, for tests of its host
// side without a GPU: buffers are host buffers, copies copy, kernels are
// recorded by name and launch shape but do not run, and hipMalloc can be made to
// fail, once or from some call on. Loaded with global symbols before the
// library, whose calls then bind here.
#include <hip/hip_runtime_api.h>

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
std::map<const void*, std::string>& names() {
  static std::map<const void*, std::string> m;
  return m;
}
std::map<const void*, size_t>& symbols() {
  static std::map<const void*, size_t> m;
  return m;
}
std::vector<Launch> launches;
long fail_in = -1;  // hipMalloc calls until one fails, -1: none does
bool fail_on;       // and every later one
size_t allocated = 0;
struct {
  dim3 grid, block;
  size_t shared;
  hipStream_t stream;
} call;
int handle;
}  // namespace

extern "C" {

void host_hip_fail_malloc(long after, int on) {
  fail_in = after;
  fail_on = on != 0;
}
void host_hip_clear() {
  launches.clear();
  allocated = 0;
}
size_t host_hip_allocated() { return allocated; }
// "name gx gy bx" per launch, one a line
size_t host_hip_launches(char* out, size_t cap) {
  std::string s;
  for (const Launch& l : launches)
    s += l.name + " " + std::to_string(l.grid.x) + " " + std::to_string(l.grid.y) + " " +
         std::to_string(l.block.x) + "\n";
  if (out && cap > s.size()) std::memcpy(out, s.c_str(), s.size() + 1);
  return s.size() + 1;
}

void** __hipRegisterFatBinary(const void*) { return reinterpret_cast<void**>(&handle); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*,
                           void*, dim3*, dim3*, int*) {
  names()[host] = name;
}
void __hipRegisterVar(void**, void* var, char*, const char*, int, size_t size, int, int) {
  symbols()[var] = size;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t shared, hipStream_t s) {
  call = {g, b, shared, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* shared, hipStream_t* s) {
  *g = call.grid;
  *b = call.block;
  *shared = call.shared;
  *s = call.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t, hipStream_t) {
  launches.push_back({names()[f], g, b});
  return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t n) {
  if (fail_in == 0) {
    if (!fail_on) fail_in = -1;
    return hipErrorOutOfMemory;
  }
  if (fail_in > 0) --fail_in;
  allocated += n;
  *p = std::calloc(n ? n : 1, 1);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = std::calloc(n ? n : 1, 1);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  std::memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) {
  return hipMemcpy(d, s, n, k);
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* var) {
  static std::map<const void*, void*> at;
  if (!at[var]) at[var] = std::calloc(symbols()[var], 1);
  *p = at[var];
  return hipSuccess;
}

hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
  std::memset(p, 0, sizeof *p);
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "host test error"; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(&handle);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = reinterpret_cast<hipEvent_t>(&handle);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 0.0f;
  return hipSuccess;
}

}  // extern "C"
