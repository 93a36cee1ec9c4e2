// pinned_on_device against a stand-in for the runtime's pointer queries: pinned
// allocations [base, base + size) whose device addresses are `shift` above the host
// ones (0: the same addresses), everything else pageable.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <vector>

struct Alloc {
  uintptr_t base;
  size_t size;
};
static std::vector<Alloc> g_allocs;
static uintptr_t g_shift;

static const Alloc *find(uintptr_t host) {
  for (const Alloc &a : g_allocs)
    if (host >= a.base && host < a.base + a.size) return &a;
  return nullptr;
}
static hipError_t fake_attributes(hipPointerAttribute_t *out, const void *p) {
  *out = hipPointerAttribute_t{};
  if (!find((uintptr_t)p)) return hipErrorInvalidValue;
  out->type = hipMemoryTypeHost;
  out->hostPointer = const_cast<void *>(p);
  out->devicePointer = (void *)((uintptr_t)p + g_shift);
  return hipSuccess;
}
static hipError_t fake_range(hipDeviceptr_t *base, size_t *size, hipDeviceptr_t d) {
  const Alloc *a = find((uintptr_t)d - g_shift);
  if (!a) return hipErrorInvalidValue;
  *base = (hipDeviceptr_t)(a->base + g_shift);
  *size = a->size;
  return hipSuccess;
}
static hipError_t fake_last() { return hipSuccess; }
#define hipPointerGetAttributes fake_attributes
#define hipMemGetAddressRange fake_range
#define hipGetLastError fake_last
#include "../../su2_amd/csrc/su2_pinned.hpp"

int main() {
  for (uintptr_t shift : {(uintptr_t)0, (uintptr_t)1 << 40}) {
    g_shift = shift;
    // two pinned allocations with a pageable page between them, and one right behind
    g_allocs = {{0x10000, 0x1000}, {0x12000, 0x1000}, {0x13000, 0x800}};
    auto at = [&](uintptr_t p, size_t n) {
      return (uintptr_t)su2k::pinned_on_device((double *)p, n);
    };
    if (at(0x10000, 0x1000) != 0x10000 + shift) return 1;   // the whole allocation
    if (at(0x10018, 0x18) != 0x10018 + shift) return 2;     // inside it
    if (at(0x10ff8, 8) != 0x10ff8 + shift) return 3;        // its end
    if (at(0x10ff8, 16) != 0) return 4;                     // past its end
    if (at(0x10000, 0x3000) != 0) return 5;                 // over the pageable page
    if (at(0x12800, 0x1000) != 0) return 6;                 // into the next allocation
    if (at(0x11000, 8) != 0 || at(0x20000, 8) != 0) return 7;  // pageable
    if (at(0x11ff8, 16) != 0) return 8;                     // from pageable into pinned
  }
  printf("ok\n");
  return 0;
}
