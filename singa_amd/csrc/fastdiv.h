// Division by a run-time constant without the division: the kernels that unflatten an index divide by plane and row sizes that
// are the same for a whole launch.
#ifndef SINGA_AMD_CSRC_FASTDIV_H_
#define SINGA_AMD_CSRC_FASTDIV_H_

#include <hip/hip_runtime.h>

// n / d for 0 <= n < 2^31, d >= 1: q = (mulhi(n, m) + n) >> s, prepared on the host
struct sgh_fastdiv {
  unsigned d, m, s;
  explicit sgh_fastdiv(unsigned d_ = 1) : d(d_), m(0), s(0) {
    while ((1ull << s) < d) ++s;
    m = unsigned(((1ull << 32) * ((1ull << s) - d)) / d + 1);
  }
  __device__ __forceinline__ int div(int n) const { return int((__umulhi(unsigned(n), m) + unsigned(n)) >> s); }
};

#endif  // SINGA_AMD_CSRC_FASTDIV_H_
