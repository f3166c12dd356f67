/*
 * dbuf.h -- a device array of a recall handle.
 */
#ifndef GSBN_DBUF_H
#define GSBN_DBUF_H

#include <hip/hip_runtime.h>

#include <cstddef>

#include "../../include/gsbn_amd.h"

/* n elements at p; none (p null, n 0) before an allocation and after one that
 * failed, so that either may be asked whether the array has to be made */
template <typename T>
struct DBuf {
  T* p = nullptr;
  size_t n = 0;
  DBuf() {}
  DBuf(const DBuf&) = delete;
  DBuf& operator=(const DBuf&) = delete;
  ~DBuf() {
    if (p) (void)hipFree(p);
  }
  hipError_t alloc(size_t count) {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
    if (!count) return hipSuccess;
    hipError_t e = hipMalloc(&p, count * sizeof(T));
    if (e != hipSuccess) {
      /* once more without the memory that closed solvers left */
      (void)hipGetLastError();
      (void)gsbn_memory_release();
      e = hipMalloc(&p, count * sizeof(T));
    }
    if (e != hipSuccess) {
      (void)hipGetLastError();
      p = nullptr;
      return e;
    }
    n = count;
    return hipSuccess;
  }
  hipError_t upload(const T* h, size_t count) {
    hipError_t e = alloc(count);
    if (e == hipSuccess && count) e = hipMemcpy(p, h, count * sizeof(T), hipMemcpyHostToDevice);
    return e;
  }
};

#endif /* GSBN_DBUF_H */
