// su2_pinned.hpp -- whether a kernel may write a host range.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace su2k {

// The device address of the host range [p, p + bytes), or null: all of it has to lie
// in one pinned allocation.  Asked of the allocation itself: equal distances of two
// addresses on host and device say nothing where both are the same addresses, as they
// are here, so a range whose ends are pinned in two allocations would pass.
inline double *pinned_on_device(double *p, size_t bytes) {
  hipPointerAttribute_t a;
  hipDeviceptr_t base = nullptr;
  size_t size = 0;
  if (bytes == 0 || hipPointerGetAttributes(&a, p) != hipSuccess || a.type != hipMemoryTypeHost ||
      !a.devicePointer ||
      hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)a.devicePointer) != hipSuccess) {
    (void)hipGetLastError();  // pageable memory: not an error here
    return nullptr;
  }
  const char *d = (const char *)a.devicePointer, *b = (const char *)base;
  if (!b || d < b || (size_t)(d - b) > size || bytes > size - (size_t)(d - b)) return nullptr;
  return (double *)a.devicePointer;
}

}  // namespace su2k
