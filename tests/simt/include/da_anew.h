// Stand-in for csrc/da_anew.h on the CPU, where nothing is held in registers.
#pragma once

template <typename T>
static inline T da_anew(T v) { return v; }
