// Stand-in for csrc/da_read_arg.h on the CPU, where an argument is there already.
#pragma once

template <typename T>
static inline void da_read_arg(T) {}
