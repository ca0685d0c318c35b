// Compares DivBounded's quotients with n / d, bit for bit, on the device: kind 0
// operands of random mantissas and signs over the whole range of slopes, kind 1 divisors
// just below a power of two and kind 2 random divisors, both with numerators within
// a unit of their last place of those whose quotient is halfway between two
// values, where rounding is closest.  Built into a library of its own for
// test_gpu_quotients.py.
#include "sweep_dev.h"

namespace {

__device__ unsigned long long mix(unsigned long long x) {  // splitmix64
  x += 0x9e3779b97f4a7c15ull;
  x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
  x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
  return x ^ (x >> 31);
}

__device__ double value(unsigned long long mantissa, int exponent, unsigned long long sign) {
  return __builtin_bit_cast(double, sign << 63 | (unsigned long long)(1023 + exponent) << 52 |
                                        (mantissa & 0xfffffffffffffull));
}

__global__ void k_check(int kind, long count, unsigned long long seed, unsigned long long *out) {
  const long step = (long)gridDim.x * blockDim.x;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += step) {
    const unsigned long long a = mix(seed + 2 * i), b = mix(seed + 2 * i + 1);
    double n, d;
    if (kind == 0) {  // exponents -73 .. 763
      d = value(a, (int)(a >> 52) % 837 - 73, b >> 63);
      n = value(b, (int)(b >> 52 & 0x7ff) % 837 - 73, a >> 63);
    } else {
      d = kind == 1 ? 2.0 - (double)(i + 1) * 0x1p-52 : value(a, 0, 0);
      const double q = value(b, 0, 0);
      n = __builtin_fma(d, q, d * 0x1p-53);
    }
    for (int k = kind == 0 ? 0 : -1; k <= (kind == 0 ? 0 : 1); ++k) {
      const double m = __builtin_bit_cast(double, __builtin_bit_cast(unsigned long long, n) + k);
      le2d::DivBounded dv;
      const unsigned long long got = __builtin_bit_cast(unsigned long long, dv.ratio(m, d));
      if (got != __builtin_bit_cast(unsigned long long, m / d) && atomicAdd(out, 1ull) == 0) {
        out[1] = __builtin_bit_cast(unsigned long long, m);
        out[2] = __builtin_bit_cast(unsigned long long, d);
      }
    }
  }
}

}  // namespace

// out: pairs that differ, then one of them (bits of n and d).  Returns a HIP error.
extern "C" int check_quotients(int kind, long count, unsigned long long seed,
                               unsigned long long out[3]) {
  unsigned long long *d = nullptr;
  hipError_t e = hipMalloc(&d, 3 * sizeof *d);
  if (e != hipSuccess) return e;
  e = hipMemset(d, 0, 3 * sizeof *d);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_check, dim3(8192), dim3(256), 0, nullptr, kind, count, seed, d);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpy(out, d, 3 * sizeof *d, hipMemcpyDeviceToHost);
  (void)hipFree(d);
  return e;
}
