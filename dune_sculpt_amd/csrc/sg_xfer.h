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

int sg_set_error(const char *fmt, ...);
int sg_check_hip(hipError_t e, const char *what);
