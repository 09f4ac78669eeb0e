// Check of near_math.h's square root, reciprocal and quotient against the IEEE
// forms on the GPU at hand: their exactness rests on the hardware's
// approximations, so it is measured rather than assumed.
#include "near_math.h"

namespace dsph {

__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  // splitmix64's finalizer (Steele, Lea, Flood: "Fast splittable pseudorandom
  // number generators", OOPSLA 2014)
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

// 2^e (1 + m / 2^23)
__device__ __forceinline__ float make_f32(int e, uint32_t m) {
  return __uint_as_float(((uint32_t)(e + 127) << 23) | (m & 0x7fffffu));
}

__global__ void __launch_bounds__(kBlock) k_near_check(int op, uint32_t first, int64_t n, uint64_t seed,
                                                       unsigned long long* __restrict__ differ) {
  unsigned long long bad = 0;
  const int64_t step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += step) {
    const float x = __uint_as_float(first + (uint32_t)i);
    float got, ref;
    if (op == 0) {
      got = sqrt_near(x);
      ref = sqrt_rn(x);
    } else if (op == 1) {
      got = rcp_near(x);
      ref = 1.0f / x;
    } else {
      // exponents over the whole range, every fourth mantissa near 1 or 2, where
      // the hard cases of a quotient lie
      const uint64_t z = mix64(seed + (uint64_t)i * 0x9e3779b97f4a7c15ull);
      uint32_t ma = (uint32_t)z, mb = (uint32_t)(z >> 23);
      if ((i & 3) == 1) ma &= 15u;
      if ((i & 3) == 2) mb = ~(mb & 15u);
      const float a = make_f32(-40 + (int)((z >> 46) % 98), ma), b = make_f32(-58 + (int)((z >> 53) % 116), mb);
      const float s = (z >> 63) ? -a : a;
      got = div_near(s, b, rcp_near(b));
      ref = s / b;
    }
    bad += __float_as_uint(got) != __float_as_uint(ref) ? 1u : 0u;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) bad += __shfl_xor(bad, o, 64);
  if ((threadIdx.x & 63) == 0 && bad) atomicAdd(differ, bad);
}

}  // namespace dsph

using namespace dsph;

extern "C" int dsph_near_check(int32_t op, uint32_t first, int64_t n, uint64_t seed, int64_t* differ, void* stream) {
  if (op < 0 || op > 2 || n < 0 || !differ) return DSPH_ERR_ARG;
  if (op < 2 && n > ((int64_t)1 << 32) - first) return DSPH_ERR_ARG;
  if (n == 0) return DSPH_OK;
  k_near_check<<<4096, kBlock, 0, as_stream(stream)>>>(op, first, n, seed,
                                                       reinterpret_cast<unsigned long long*>(differ));
  return launch_status();
}
