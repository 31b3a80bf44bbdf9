// n / d by a multiplication, for a divisor that the host knows and 0 <= n < 2^31: with
// l = ceil(log2 d) and mul = ceil(2^(31+l) / d), mul·d exceeds 2^(31+l) by less than
// d <= 2^l, so n·mul / 2^(31+l) exceeds n/d by less than 1/d. (Granlund and Montgomery,
// Division by Invariant Integers using Multiplication, 1994.)
#pragma once

#include <stdint.h>

#ifdef __HIPCC__
#define BVLLM_HOST_DEVICE __host__ __device__
#else
#define BVLLM_HOST_DEVICE
#endif

namespace bvllm {

struct FastDiv {
  uint32_t mul, shift;
  BVLLM_HOST_DEVICE int32_t operator()(int32_t n) const { return (int32_t)(((uint64_t)(uint32_t)n * mul) >> shift); }
};

inline FastDiv fast_div(int32_t d) {
  uint32_t l = 0;
  while (((int64_t)1 << l) < d) ++l;
  return {(uint32_t)((((uint64_t)1 << (31 + l)) + (uint64_t)d - 1) / (uint64_t)d), 31 + l};
}

}  // namespace bvllm
