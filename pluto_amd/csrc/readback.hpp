// Arrays of a domain or a patch to the caller's host memory (readback.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace pgpu {

// What is read: na device arrays, of each the n[0] x n[1] x n[2] cells from
// element `first` on with row and plane strides, x fastest.
struct ReadSrc {
  const double* a[11];
  int na = 0;
  int n[3] = {0, 0, 0};
  long first = 0, row = 0, plane = 0;
};

// Pinned staging of an object's read-backs: a ring of buffers, made at the
// first one, replaced by larger ones for a larger read, and kept with the object.
struct Readback {
  static constexpr int NB = 4;
  double* h[NB] = {nullptr, nullptr, nullptr, nullptr};
  hipEvent_t ev[NB] = {nullptr, nullptr, nullptr, nullptr};
  long elems = 0;   // doubles of one buffer
  ~Readback();
};

// Copies src's arrays to dst[0 .. na-1] (n cells each) after what stream s
// holds; returns when they are there.  A hipError_t (0: done).
int readback(Readback& rb, const ReadSrc& src, double* const* dst, hipStream_t s);

}  // namespace pgpu
