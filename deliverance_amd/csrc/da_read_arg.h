// Reads a kernel argument and drops it: its word is asked for here and not where it is used, which may be a
// round trip later (an argument's line of memory is seldom in a cache when its kernel starts).
#pragma once
#include <hip/hip_runtime.h>

template <typename T>
__device__ __forceinline__ void da_read_arg(T v) { asm volatile("" ::"s"(v)); }
