// A number as if it were new: what is worked out from it is worked out behind this line, and not in front of it (of a loop above all)
// to be held in vector registers until it is used.
#pragma once
#include <hip/hip_runtime.h>

template <typename T>
__device__ __forceinline__ T da_anew(T v) {
  asm volatile("" : "+v"(v));
  return v;
}
