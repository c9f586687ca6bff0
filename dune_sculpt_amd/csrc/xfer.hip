// Several copies as one launch.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "sg_xfer.h"

// Bound by HBM for large meshes and by the launch for small ones.  A checkpoint is 13 to 17
// arrays: as one hipMemcpyAsync each they took 4 to 10 us of host time apiece.  One launch
// takes a workgroup per COPY_CHUNK bytes over all of them, 16 bytes per lane (4 where an
// address is not a multiple of 16), four loads ahead of the stores.
#define COPY_CHUNK 16384

namespace {
struct CopyArgs {
  SgCopy c[SG_COPY_MAX];
  int first[SG_COPY_MAX + 1];  // first workgroup of each copy
  int n;
};

template <class T>
__device__ __forceinline__ void copy_chunk(char *dst, const char *src, size_t bytes) {
  T *d = (T *)dst;
  const T *s = (const T *)src;
  const int n = (int)(bytes / sizeof(T)), t = threadIdx.x;
  for (int i = t; i < n; i += 4 * 256) {
    T v[4];
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = s[min(i + q * 256, n - 1)];
#pragma unroll
    for (int q = 0; q < 4; q++)
      if (i + q * 256 < n) d[i + q * 256] = v[q];
  }
}

__global__ __launch_bounds__(256) void k_copies(CopyArgs a) {
  int i = 0;
  while (i + 1 < a.n && (int)blockIdx.x >= a.first[i + 1]) i++;
  const size_t off = (size_t)((int)blockIdx.x - a.first[i]) * COPY_CHUNK;
  char *d = (char *)a.c[i].dst + off;
  const char *s = (const char *)a.c[i].src + off;
  const size_t n = min((size_t)COPY_CHUNK, a.c[i].bytes - off);
  if ((((uintptr_t)d | (uintptr_t)s | n) & 15) == 0)
    copy_chunk<int4>(d, s, n);
  else
    copy_chunk<int>(d, s, n);
}
}  // namespace

int sg_enqueue_copies(hipStream_t s, const SgCopy *c, int n) {
  CopyArgs a;
  a.n = 0;
  a.first[0] = 0;
  auto flush = [&]() -> int {
    if (a.n == 0) return 0;
    hipLaunchKernelGGL(k_copies, dim3(a.first[a.n]), dim3(256), 0, s, a);
    a.n = 0;
    return sg_check_hip(hipGetLastError(), "copy launch");
  };
  for (int i = 0; i < n; i++) {
    if (c[i].bytes == 0) continue;
    if (((uintptr_t)c[i].dst | (uintptr_t)c[i].src | c[i].bytes) & 3) return sg_set_error("copy: not 4-byte aligned");
    const size_t blocks = (c[i].bytes + COPY_CHUNK - 1) / COPY_CHUNK;
    if (blocks > (1u << 30)) return sg_set_error("copy: too large");
    if (a.n == SG_COPY_MAX || (size_t)a.first[a.n] + blocks > (1u << 30))
      if (int rc = flush()) return rc;
    a.c[a.n] = c[i];
    a.first[a.n + 1] = a.first[a.n] + (int)blocks;
    a.n++;
  }
  return flush();
}
