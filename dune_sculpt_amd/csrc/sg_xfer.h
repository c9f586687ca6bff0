// Several copies as one launch (xfer.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

#define SG_COPY_MAX 24  // copies per launch

struct SgCopy {  // sizes and addresses are multiples of 4
  void *dst;
  const void *src;
  size_t bytes;
};
// The copies as one launch (more than SG_COPY_MAX: one per SG_COPY_MAX); ranges that
// overlap are the caller's error.
int sg_enqueue_copies(hipStream_t s, const SgCopy *c, int n);

// Pinned host memory of a PBVH or batch for the copies of its host-driven calls: grow-only,
// at most SG_PINNED_MAX bytes, freed with its owner.  Every user waits for the stream before
// it returns, so the next one finds it idle.
#define SG_PINNED_MAX ((size_t)2 << 20)
struct SgPinned {
  void *host = nullptr;
  size_t cap = 0;
};
void *sg_pinned(SgPinned &b, size_t bytes);  // null: larger than SG_PINNED_MAX, or no memory
void sg_pinned_free(SgPinned &b);
// Device memory to the caller's host memory, waited for (4-byte aligned, as SgCopy).
int sg_read_back(hipStream_t s, SgPinned &b, const void *dev, void *out, size_t bytes, const char *what);
int sg_enqueue_zero(hipStream_t s, int *p, int n);

int sg_set_error(const char *fmt, ...);
int sg_check_hip(hipError_t e, const char *what);
