// The record buffers of a handle under a failing allocator (capi.cpp's alloc_records, host only): a
// call that fails leaves nothing that a later call takes for a whole set.
//
// Usage: alloc_records; exit 0 when every case holds
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>

static int calls, fail_at;
template <class T>
static hipError_t test_malloc(T **p, size_t) {
  if (calls++ == fail_at) return hipErrorOutOfMemory;
  *p = static_cast<T *>(std::malloc(8));
  return hipSuccess;
}
#define hipMalloc test_malloc
#include "capi.cpp"
#undef hipMalloc

int main() {
  for (int dim = 2; dim <= 3; ++dim)
    for (int k = 0; k < 3; ++k) {
      ppk_mhd_solver h;
      h.dp = {};
      h.dp.dim = dim;
      calls = 0;
      fail_at = k;
      if (alloc_records(&h)) return std::printf("%dD: allocation %d failed, call did not\n", dim, k), 1;
      fail_at = -1;
      if (!alloc_records(&h)) return std::printf("%dD: second call failed\n", dim), 1;
      if (!h.fw.rec || !h.fw.flux || !h.fw.emf)
        return std::printf("%dD: a buffer is missing after allocation %d failed once\n", dim, k), 1;
      if (calls != 4) return std::printf("%dD: %d allocations for three buffers\n", dim, calls), 1;
    }
  return 0;
}
