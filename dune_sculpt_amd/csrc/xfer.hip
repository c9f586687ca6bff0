// Several copies as one launch, and pinned host memory of a PBVH or batch.
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

__global__ __launch_bounds__(256) void k_zero(int *p, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0;
}
}  // namespace

int sg_enqueue_zero(hipStream_t s, int *p, int n) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(k_zero, dim3(std::min((n + 255) / 256, 1024)), dim3(256), 0, s, p, n);
  return sg_check_hip(hipGetLastError(), "clear launch");
}

void *sg_pinned(SgPinned &b, size_t bytes) {
  if (bytes > SG_PINNED_MAX) return nullptr;
  if (bytes <= b.cap) return b.host;
  sg_pinned_free(b);
  size_t cap = (size_t)512 << 10;  // few growths: pinning costs about as much as the call it serves
  while (cap < bytes) cap *= 2;
  if (hipHostMalloc(&b.host, cap, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    b.host = nullptr;
    return nullptr;
  }
  b.cap = cap;
  return b.host;
}

void sg_pinned_free(SgPinned &b) {
  if (b.host) (void)hipHostFree(b.host);
  b = SgPinned();
}

// Up to SG_PINNED_MAX a copy kernel into pinned memory and a memcpy; hipMemcpyAsync into
// pageable memory stages the same bytes in pieces with a wait each, which pays for larger
// sizes only.  Positions and normals of 32 meshes (650 k vertices), a call each: 0.23 ms
// less.
int sg_read_back(hipStream_t s, SgPinned &b, const void *dev, void *out, size_t bytes, const char *what) {
  void *h = sg_pinned(b, bytes);
  if (!h) {
    if (int rc = sg_check_hip(hipMemcpyAsync(out, dev, bytes, hipMemcpyDeviceToHost, s), what)) return rc;
    return sg_check_hip(hipStreamSynchronize(s), what);
  }
  const SgCopy c = {h, dev, bytes};
  if (int rc = sg_enqueue_copies(s, &c, 1)) return rc;
  if (int rc = sg_check_hip(hipStreamSynchronize(s), what)) return rc;
  memcpy(out, h, bytes);
  return 0;
}

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
