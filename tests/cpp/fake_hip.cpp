// A HIP runtime in host memory, for tests of the host code without a GPU: it
// stands in for libamdhip64 when loaded first with global symbols.  Streams run
// in order at once, kernels are counted by name and not run, and an allocation
// can be made to fail.
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

namespace {
struct Dim3 {
  unsigned x, y, z;
};
constexpr int kSuccess = 0, kInvalidValue = 1, kOutOfMemory = 2;
std::mutex mu;
std::map<const void*, std::string>& names() {  // filled while other libraries are loaded
  static std::map<const void*, std::string> m;
  return m;
}
std::map<std::string, int> launches;
int fail_in = 0, copies_to_host = 0;
char symbol[1 << 20];
}  // namespace

extern "C" {

// The n-th allocation of device memory from now on fails (0: none).
void fake_fail_malloc(int n) { fail_in = n; }
// Launches of kernels whose name contains `part`, and copies to the host, since the last reset.
int fake_launches(const char* part) {
  int n = 0;
  for (const auto& l : launches)
    if (l.first.find(part) != std::string::npos) n += l.second;
  return n;
}
int fake_copies_to_host() { return copies_to_host; }
void fake_reset() {
  launches.clear();
  copies_to_host = 0;
}

int hipMalloc(void** p, size_t n) {
  if (fail_in > 0 && --fail_in == 0) return kOutOfMemory;
  *p = std::malloc(n ? n : 1);
  return *p ? kSuccess : kOutOfMemory;
}
int hipFree(void* p) {
  std::free(p);
  return kSuccess;
}
int hipHostMalloc(void** p, size_t n, unsigned) {
  *p = std::malloc(n);
  return *p ? kSuccess : kOutOfMemory;
}
int hipHostFree(void* p) {
  std::free(p);
  return kSuccess;
}
int hipMemcpyAsync(void* dst, const void* src, size_t n, int kind, void*) {
  std::memcpy(dst, src, n);
  const std::lock_guard<std::mutex> lock(mu);
  copies_to_host += kind == 2;
  return kSuccess;
}
int hipMemsetAsync(void* p, int v, size_t n, void*) {
  std::memset(p, v, n);
  return kSuccess;
}
int hipMemsetD32Async(void* p, int v, size_t n, void*) {
  for (size_t i = 0; i < n; ++i) std::memcpy((char*)p + 4 * i, &v, 4);
  return kSuccess;
}
int hipPointerGetAttributes(void*, const void*) { return kInvalidValue; }  // memory HIP does not know
int hipMemGetInfo(size_t* free, size_t* total) {
  *free = *total = (size_t)8 << 30;
  return kSuccess;
}
int hipGetSymbolAddress(void** p, const void*) {
  *p = symbol;
  return kSuccess;
}
int hipSetDevice(int) { return kSuccess; }
int hipGetDevice(int* d) {
  *d = 0;
  return kSuccess;
}
int hipGetDeviceCount(int* n) {
  *n = 1;
  return kSuccess;
}
int hipDeviceGetAttribute(int* v, int, int) {
  *v = 256;
  return kSuccess;
}
int hipGetLastError() { return kSuccess; }
const char* hipGetErrorString(int) { return "fake error"; }
int hipStreamCreateWithFlags(void** s, unsigned) {
  *s = symbol;
  return kSuccess;
}
int hipStreamDestroy(void*) { return kSuccess; }
int hipStreamSynchronize(void*) { return kSuccess; }
int hipStreamWaitEvent(void*, void*, unsigned) { return kSuccess; }
int hipEventCreate(void** e) {
  *e = symbol;
  return kSuccess;
}
int hipEventCreateWithFlags(void** e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void*) { return kSuccess; }
int hipEventRecord(void*, void*) { return kSuccess; }
int hipEventQuery(void*) { return kSuccess; }
int hipEventSynchronize(void*) { return kSuccess; }
int hipEventElapsedTime(float* ms, void*, void*) {
  *ms = 0;
  return kSuccess;
}

int hipLaunchKernel(const void* f, Dim3, Dim3, void**, size_t, void*) {
  const std::lock_guard<std::mutex> lock(mu);
  ++launches[names()[f]];
  return kSuccess;
}
int __hipPushCallConfiguration(Dim3, Dim3, size_t, void*) { return kSuccess; }
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* lds, void** stream) {
  *grid = *block = Dim3{1, 1, 1};
  *lds = 0;
  *stream = nullptr;
  return kSuccess;
}
void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  names()[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}

}  // extern "C"
