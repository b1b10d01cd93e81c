// Compares root() and quotients() of csrc/contact_math.h with sqrtf and the
// division, bit for bit, on the GPU.
#include <cstdint>

#include "contact_math.h"

namespace {

__device__ inline float of(uint32_t b) { return __uint_as_float(b); }

// [0] floats whose root differs, [1] floats whose y is further than 2^-20 off
// (or, outside [2^-96, 2^96], is not NaN).
__global__ __launch_bounds__(256) void k_root(uint32_t first, uint64_t count, unsigned long long* out) {
  const uint64_t stride = (uint64_t)gridDim.x * 256u;
  unsigned long long wrong = 0, far = 0;
  for (uint64_t i = blockIdx.x * 256u + threadIdx.x; i < count; i += stride) {
    const float x = of(first + (uint32_t)i), want = sqrtf(x);
    float y;
    const float got = dem::root(x, y);
    wrong += __float_as_uint(got) != __float_as_uint(want) && !(got != got && want != want);
    const bool inside = x >= 0x1p-96f && x <= 0x1p96f;
    far += inside ? !(fabs((double)y * sqrt((double)x) - 1.0) <= 0x1p-20) : y == y;
  }
  if (wrong) atomicAdd(&out[0], wrong);
  if (far) atomicAdd(&out[1], far);
}

__device__ inline uint32_t mix(uint64_t k) {  // splitmix64's finalizer
  k = (k ^ (k >> 30)) * 0xBF58476D1CE4E5B9ull;
  k = (k ^ (k >> 27)) * 0x94D049BB133111EBull;
  return (uint32_t)((k ^ (k >> 31)) >> 16);
}

// Quotients a / b and c / b for b and y as root() returns them.  kHard: a is
// one of the floats around a midpoint of two floats times b, so the quotient
// is as near to a midpoint as it gets; else a is any float at all, c any with
// an exponent near b's.
template <bool kHard>
__global__ __launch_bounds__(256) void k_quotients(uint64_t seed, uint64_t count, unsigned long long* out) {
  const uint64_t stride = (uint64_t)gridDim.x * 256u;
  unsigned long long wrong = 0;
  for (uint64_t i = blockIdx.x * 256u + threadIdx.x; i < count; i += stride) {
    const uint64_t k = (seed + i) * 0x9E3779B97F4A7C15ull;
    const uint32_t r0 = mix(k), r1 = mix(k + 1u), r2 = mix(k + 2u), r3 = mix(k + 3u);
    // x in [2^-96, 2^96)
    const float x = of(((31u + r0 % 192u) << 23) | (r1 & 0x7FFFFFu));
    float y;
    const float b = dem::root(x, y);
    float a, c;
    if (kHard) {
      const uint32_t q = ((97u + r2 % 61u) << 23) | (r3 & 0x7FFFFFu);
      const double mid = 0.5 * ((double)of(q) + (double)of(q + 1u));
      a = (float)(mid * (double)b);
      c = of(__float_as_uint(a) + 1u - 2u * (r0 >> 31));
    } else {
      a = of(r2 ^ (r3 << 16));
      c = of((r3 & 0x807FFFFFu) | ((__float_as_uint(b) + ((r1 >> 23 & 31u) - 16u << 23)) & 0x7F800000u));
    }
    float qa, qc;
    dem::quotients(a, c, b, y, qa, qc);
    const float wa = a / b, wc = c / b;
    wrong += __float_as_uint(qa) != __float_as_uint(wa) && !(qa != qa && wa != wa);
    wrong += __float_as_uint(qc) != __float_as_uint(wc) && !(qc != qc && wc != wc);
  }
  if (wrong) atomicAdd(&out[0], wrong);
}

template <class Launch>
int counted(uint64_t out[2], Launch&& launch) {
  unsigned long long* d = nullptr;
  hipError_t e = hipMalloc((void**)&d, 16);
  if (e == hipSuccess) e = hipMemset(d, 0, 16);
  if (e == hipSuccess) {
    launch(d);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpy(out, d, 16, hipMemcpyDeviceToHost);
  if (d) (void)hipFree(d);
  return (int)e;
}

}  // namespace

// Each returns a hipError_t.
extern "C" int check_root(uint32_t first, uint64_t count, uint64_t out[2]) {
  return counted(out, [&](unsigned long long* d) { k_root<<<4096, 256>>>(first, count, d); });
}

extern "C" int check_quotients(int hard, uint64_t seed, uint64_t count, uint64_t out[2]) {
  return counted(out, [&](unsigned long long* d) {
    if (hard) k_quotients<true><<<4096, 256>>>(seed, count, d);
    else k_quotients<false><<<4096, 256>>>(seed, count, d);
  });
}
