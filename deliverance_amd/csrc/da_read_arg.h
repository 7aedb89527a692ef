// Reads a kernel argument and drops it: the compiler asks for its word with the other arguments.  Why a kernel would want that stands
// where it does (gemm_mfma.hip).
#pragma once
#include <hip/hip_runtime.h>

template <typename T>
__device__ __forceinline__ void da_read_arg(T v) { asm volatile("" ::"s"(v)); }
