// Device memory and synchronisation plumbing for hosts that bind the C ABI without a HIP
// runtime of their own (Python via ctypes, Fortran via iso_c_binding).  Keeping these in the
// library means a process loads exactly one HIP runtime: the one libself_amd.so links.
#include "selfamd_common.hpp"
#include "../../include/self_amd.h"

using namespace selfamd;

namespace selfamd {

Source source_of(const void *p, size_t bytes, size_t align, int device) {
  hipPointerAttribute_t at{};
  auto known = [&](const void *q) {
    const hipError_t e = hipPointerGetAttributes(&at, q);
    if (e != hipSuccess) (void)hipGetLastError();  // memory that the runtime does not know
    return e == hipSuccess && at.type != hipMemoryTypeUnregistered;
  };
  if (!known(p) || at.type != hipMemoryTypeDevice) return Source::kCopy;
  const int owner = at.device;
  hipDeviceptr_t base = nullptr;
  size_t size = 0;
  if (hipMemGetAddressRange(&base, &size, const_cast<void *>(p)) != hipSuccess) {
    (void)hipGetLastError();
    return Source::kCopy;
  }
  const size_t before = reinterpret_cast<uintptr_t>(p) - reinterpret_cast<uintptr_t>(base);
  if (before <= size && bytes <= size - before)
    return owner == device && reinterpret_cast<uintptr_t>(p) % align == 0 ? Source::kKernel : Source::kCopy;
  return known(static_cast<const char *>(p) + bytes - 1) ? Source::kCopy : Source::kShort;
}

}  // namespace selfamd

extern "C" {

int selfamd_device_count(int *count) {
  SELFAMD_REQUIRE(count, "device_count: null argument");
  *count = 0;
  hipError_t e = hipGetDeviceCount(count);
  if (e != hipSuccess) *count = 0;
  return kOk;
}

int selfamd_device_name(int device, char *name, int len) {
  SELFAMD_REQUIRE(name && len > 0, "device_name: null argument");
  hipDeviceProp_t prop;
  SELFAMD_HIP(hipGetDeviceProperties(&prop, device));
  snprintf(name, (size_t)len, "%s (%s, %d CUs)", prop.name, prop.gcnArchName, prop.multiProcessorCount);
  return kOk;
}

int selfamd_malloc(void **ptr, size_t bytes) {
  SELFAMD_REQUIRE(ptr, "malloc: null argument");
  *ptr = nullptr;
  SELFAMD_HIP(hipMalloc(ptr, bytes ? bytes : 8));
  return kOk;
}

int selfamd_free(void *ptr) {
  if (ptr) SELFAMD_HIP(hipFree(ptr));
  return kOk;
}

int selfamd_memcpy(void *dst, const void *src, size_t bytes, int kind) {
  SELFAMD_REQUIRE(kind >= 1 && kind <= 3, "memcpy: kind %d (1 = H2D, 2 = D2H, 3 = D2D)", kind);
  if (!bytes) return kOk;
  SELFAMD_REQUIRE(dst && src, "memcpy: null pointer");
  const hipMemcpyKind k = kind == 1 ? hipMemcpyHostToDevice : kind == 2 ? hipMemcpyDeviceToHost : hipMemcpyDeviceToDevice;
  SELFAMD_HIP(hipMemcpy(dst, src, bytes, k));
  // The runtime may return from a copy whose target is device memory before the copy has landed.
  // The models' streams do not wait for the null stream, so a copy that they make of dst next
  // (set_solution, set_static) would read what the memory held before.
  if (kind != 2) SELFAMD_HIP(hipStreamSynchronize(nullptr));
  return kOk;
}

int selfamd_memset(void *ptr, int value, size_t bytes) {
  if (!bytes) return kOk;
  SELFAMD_REQUIRE(ptr, "memset: null pointer");
  SELFAMD_HIP(hipMemset(ptr, value, bytes));
  SELFAMD_HIP(hipStreamSynchronize(nullptr));  // as in selfamd_memcpy
  return kOk;
}

int selfamd_time_copy_f64(const double *src, double *dst, size_t n, int reps, double *elapsedMs) {
  SELFAMD_REQUIRE(elapsedMs && reps > 0, "time_copy_f64: bad arguments");
  hipStream_t st;
  SELFAMD_HIP(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
  hipEvent_t e0, e1;
  SELFAMD_HIP(hipEventCreate(&e0));
  SELFAMD_HIP(hipEventCreate(&e1));
  int rc = selfamd_copy_f64(src, dst, n, st);  // warm-up
  if (rc) return rc;
  SELFAMD_HIP(hipEventRecord(e0, st));
  for (int r = 0; r < reps && rc == 0; r++) rc = selfamd_copy_f64(src, dst, n, st);
  if (rc) return rc;
  SELFAMD_HIP(hipEventRecord(e1, st));
  SELFAMD_HIP(hipEventSynchronize(e1));
  float ms = 0.f;
  SELFAMD_HIP(hipEventElapsedTime(&ms, e0, e1));
  *elapsedMs = ms;
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  SELFAMD_HIP(hipStreamDestroy(st));
  return kOk;
}

int selfamd_device_synchronize(void) {
  SELFAMD_HIP(hipDeviceSynchronize());
  return kOk;
}

}  // extern "C"
