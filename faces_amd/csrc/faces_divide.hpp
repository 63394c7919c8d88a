// faces_divide.hpp -- division by a divisor known on the host.
#pragma once

#include <hip/hip_runtime.h>

namespace faces {

// Division of a non-negative 31-bit number by a divisor known on the host:
// q = x * mul >> sh with mul = ceil(2^sh / d), sh = 31 + ceil(log2 d), which
// is exact for x < 2^31 (mul * d - 2^sh < d <= 2^(sh-31)).  A division by a
// run-time divisor is a chain of about 30 dependent instructions, four of
// them before an item's first load.
struct Divide {
  unsigned mul;
  int sh;
  __host__ __device__ int operator()(int x) const { return (int)(((unsigned long long)(unsigned)x * mul) >> sh); }
};

inline Divide divide_by(int d)
{
  int lg = 0;
  while ((1L << lg) < d) lg++;
  Divide v;
  v.sh = 31 + lg;
  v.mul = (unsigned)(((1ULL << v.sh) + (unsigned)d - 1) / (unsigned)d);
  return v;
}

}  // namespace faces
