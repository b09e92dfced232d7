// A HIP runtime without a device, for the tests of the library's host code: device memory is host memory under a
// limit that the test sets, kernels do nothing.  Test infrastructure only; loaded before the library, whose calls
// it then serves.
#include <stddef.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <unordered_map>

namespace {
std::unordered_map<void*, size_t> sizes;
size_t used = 0, limit = SIZE_MAX;
int64_t mallocs = 0;
int last_error = 0;
char symbol[1 << 26];
}  // namespace

extern "C" {
size_t fake_used() { return used; }
void fake_limit(size_t bytes) { limit = bytes; }
int64_t fake_mallocs() { return mallocs; }

int hipMalloc(void** p, size_t n) {
  ++mallocs;
  if (n > limit || used > limit - n) {
    *p = nullptr;
    return last_error = 2;  // hipErrorOutOfMemory
  }
  *p = calloc(1, n ? n : 1);
  sizes[*p] = n;
  used += n;
  return 0;
}
int hipFree(void* p) {
  const auto it = sizes.find(p);
  if (it != sizes.end()) {
    used -= it->second;
    sizes.erase(it);
    free(p);
  }
  return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned) {
  *p = calloc(1, n);
  return 0;
}
int hipHostFree(void* p) {
  free(p);
  return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int) {
  memcpy(d, s, n);
  return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) {
  memcpy(d, s, n);
  return 0;
}
int hipMemset(void* d, int v, size_t n) {
  memset(d, v, n);
  return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void*) {
  memset(d, v, n);
  return 0;
}
int hipLaunchKernel(const void*, uint64_t, uint64_t, uint64_t, uint64_t, void**, size_t, void*) { return 0; }
int hipExtLaunchKernel(const void*, uint64_t, uint64_t, uint64_t, uint64_t, void**, size_t, void*, void*, void*, int) { return 0; }
int __hipPushCallConfiguration(uint64_t, uint64_t, uint64_t, uint64_t, size_t, void*) { return 0; }
int __hipPopCallConfiguration(void*, void*, size_t*, void**) { return 0; }
void** __hipRegisterFatBinary(const void*) { return (void**)symbol; }
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
int hipGetSymbolAddress(void** p, const void*) {
  *p = symbol;
  return 0;
}
int hipDeviceGetAttribute(int* v, int, int) {
  *v = 256;
  return 0;
}
int hipGetDevice(int* d) {
  *d = 0;
  return 0;
}
int hipDeviceSynchronize() { return 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipStreamQuery(void*) { return 0; }
int hipEventCreate(void** e) {
  *e = symbol;
  return 0;
}
int hipEventCreateWithFlags(void** e, unsigned) {
  *e = symbol;
  return 0;
}
int hipEventDestroy(void*) { return 0; }
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*) {
  *ms = 0.f;
  return 0;
}
int hipGetLastError() {
  const int e = last_error;
  last_error = 0;
  return e;
}
const char* hipGetErrorString(int) { return "fake error"; }
}
