// Reads a kernel argument and drops it: the compiler asks for its word with the other arguments.  Why a kernel would want that stands
// where it does (gemm_mfma.hip).
#pragma once
#include <hip/hip_runtime.h>

__device__ __forceinline__ void da_read_arg(int v) { asm volatile("" ::"s"(v)); }
