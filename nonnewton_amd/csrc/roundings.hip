// roundings.hip -- a check of this device: the shortened square root and division
// of device_common.h against the correctly rounded ones, bit for bit.
#include <hip/hip_runtime.h>

#include "batch.h"
#include "device_common.h"

namespace nn {

constexpr unsigned ROOT_LO = 27u << 23, ROOT_HI = 227u << 23;  // the bits of 2^-100 and 2^100
constexpr int CHECK_THREADS = 256, CHECK_BLOCKS = 4096;

__device__ __forceinline__ void count_bad(unsigned long long n, unsigned long long* bad) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) n += __shfl_xor(n, off, 64);
  if ((threadIdx.x & 63) == 0 && n) atomicAdd(bad, n);
}

// every float in [2^-100, 2^100)
__global__ __launch_bounds__(CHECK_THREADS) void k_check_roots(unsigned long long* bad) {
  unsigned long long n = 0;
  for (unsigned b = ROOT_LO + blockIdx.x * CHECK_THREADS + threadIdx.x; b < ROOT_HI; b += CHECK_THREADS * CHECK_BLOCKS) {
    const float x = __uint_as_float(b);
    n += __float_as_uint(sqrt_mid(x)) != __float_as_uint(sqrtf(x));
  }
  count_bad(n, bad);
}

// Pairs a / b with b in [2^-63, 2^52), a in [2^-100, 2^61) of either sign and a
// normal quotient: `rounds` per thread, mantissas at random and, one time in
// four each, within 4 of a power of two from above or below.
__global__ __launch_bounds__(CHECK_THREADS) void k_check_quotients(int rounds, unsigned long long* bad) {
  unsigned long long n = 0, s = 0x9E3779B97F4A7C15ull * (blockIdx.x * CHECK_THREADS + threadIdx.x + 1);
  const auto next = [&] {  // splitmix64
    s += 0x9E3779B97F4A7C15ull;
    unsigned long long z = s;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
  };
  const auto mantissa = [](unsigned r) {
    const unsigned m = r & 0x7FFFFFu, kind = r >> 30;
    return kind == 0 ? m & 3u : kind == 1 ? 0x7FFFFFu - (m & 3u) : m;
  };
  for (int r = 0; r < rounds; r++) {
    const unsigned long long u = next(), v = next();
    const unsigned ea = 27u + (unsigned)(v & 0xFFFFu) % 161u, eb = 64u + (unsigned)((v >> 16) & 0xFFFFu) % 115u;
    const float a = __uint_as_float((unsigned)(v >> 63) << 31 | ea << 23 | mantissa((unsigned)u));
    const float b = __uint_as_float(eb << 23 | mantissa((unsigned)(u >> 32)));
    if (ea + 125u < eb) continue;  // the quotient may be below the normal range
    if (ea > eb + 126u) continue;  // or above it
    n += __float_as_uint(div_mid(a, b, recip_mid(b))) != __float_as_uint(a / b);
  }
  count_bad(n, bad);
}

}  // namespace nn

extern "C" int32_t nn_check_roundings(int32_t rounds, int64_t* roots, int64_t* quotients) {
  using namespace nn;
  if (!roots || !quotients || rounds < 0 || rounds > 65536) {
    set_error("nn_check_roundings: bad arguments");
    return NN_E_ARG;
  }
  unsigned long long* bad = nullptr;
  hipError_t e = hipMalloc(&bad, 2 * sizeof(*bad));
  if (e != hipSuccess) return hip_fail(e, "nn_check_roundings: alloc");
  unsigned long long out[2] = {0, 0};
  e = hipMemcpy(bad, out, sizeof(out), hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_check_roots, dim3(CHECK_BLOCKS), dim3(CHECK_THREADS), 0, nullptr, bad);
    hipLaunchKernelGGL(k_check_quotients, dim3(CHECK_BLOCKS), dim3(CHECK_THREADS), 0, nullptr, rounds, bad + 1);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpy(out, bad, sizeof(out), hipMemcpyDeviceToHost);
  (void)hipFree(bad);
  if (e != hipSuccess) return hip_fail(e, "nn_check_roundings");
  *roots = (int64_t)out[0];
  *quotients = (int64_t)out[1];
  return NN_OK;
}
