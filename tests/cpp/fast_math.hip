// The pair loops' reciprocal, division and square root (cryo_device.hpp) against
// the IEEE operations the compiler emits, on the device: prints the number of
// results that differ, 0 0 0 expected.
//   reciprocal: every normal y up to 2^126
//   square root: every x in [2^-96, 2^126)
//   division: every significand of y; numerators 1, its neighbours, random ones,
//   and ones next to the middle between two quotients, over the stated range
#include <hip/hip_runtime.h>

#include <cstdio>

#include "cryo_device.hpp"

using namespace cryo;

constexpr unsigned kSignificands = 1u << 23;
constexpr int kThreads = 256;

__device__ float make(int exponent, unsigned significand) {
  return __uint_as_float(static_cast<unsigned>(exponent + 127) << 23 | (significand & (kSignificands - 1)));
}
__device__ unsigned mix(unsigned x) {
  x = (x ^ x >> 16) * 0x7feb352du;
  x = (x ^ x >> 15) * 0x846ca68bu;
  return x ^ x >> 16;
}
__device__ void count(unsigned long long* at, bool differs) {
  const unsigned long long lanes = __ballot(differs);
  if (differs && __ffsll(lanes) - 1 == static_cast<int>(threadIdx.x & 63))
    atomicAdd(at, static_cast<unsigned long long>(__popcll(lanes)));
}

// one thread per significand
__global__ __launch_bounds__(kThreads) void k_recip(unsigned long long* bad) {
  const unsigned m = blockIdx.x * kThreads + threadIdx.x;
  for (int e = -126; e <= 125; ++e) {
    const float y = make(e, m);
    count(&bad[0], recip_rn(y).r != 1.0f / y);
  }
  count(&bad[0], recip_rn(0x1p126f).r != 1.0f / 0x1p126f);
}
__global__ __launch_bounds__(kThreads) void k_sqrt(unsigned long long* bad) {
  const unsigned m = blockIdx.x * kThreads + threadIdx.x;
  for (int e = -96; e <= 125; ++e) {
    const float x = make(e, m);
    count(&bad[1], sqrt_rn(x) != sqrtf(x));
  }
}
__global__ __launch_bounds__(kThreads) void k_div(unsigned long long* bad) {
  const unsigned m = blockIdx.x * kThreads + threadIdx.x;
  const float y1 = make(0, m);
  auto check = [&](float x, float y) {
    const float q = x / y;
    if (!(fabsf(x) >= __uint_as_float(kFastLow)) || !(fabsf(q) >= 0x1p-126f) || !(fabsf(q) <= 0x1.fffffep127f)) return;
    count(&bad[2], div_rn(x, recip_rn(y)) != q);
  };
  check(1.0f, y1);
  check(0x1.fffffep0f, y1);
  check(y1, y1);
  for (int d = -4; d <= 4; ++d) check(__uint_as_float(__float_as_uint(y1) + d), y1);
  for (unsigned k = 0; k < 96; ++k) {
    const unsigned h = mix(m * 96u + k), g = mix(h + 0x9e3779b9u);
    const float q = make(0, h), sign = g & 1 ? -1.0f : 1.0f;
    check(sign * q, y1);
    const float mid = __builtin_fmaf(q, y1, 0x1p-24f * y1);  // next to (q + half an ulp) y
    check(mid, y1);
    check(__uint_as_float(__float_as_uint(mid) + 1), y1);
    check(__uint_as_float(__float_as_uint(mid) - 1), y1);
    // the same over the range of exponents
    const float y = make(static_cast<int>(g >> 8 & 255) % 252 - 126, m);
    check(sign * make(static_cast<int>(g >> 16 & 255) % 228 - 100, h), y);
    check(make(-100, k < 8 ? k : h), y);
  }
}

int main() {
  unsigned long long* bad = nullptr;
  unsigned long long out[3] = {0, 0, 0};
  bool ok = hipMalloc(&bad, sizeof out) == hipSuccess && hipMemcpy(bad, out, sizeof out, hipMemcpyHostToDevice) == hipSuccess;
  if (ok) {
    k_recip<<<kSignificands / kThreads, kThreads>>>(bad);
    k_sqrt<<<kSignificands / kThreads, kThreads>>>(bad);
    k_div<<<kSignificands / kThreads, kThreads>>>(bad);
    ok = hipGetLastError() == hipSuccess && hipMemcpy(out, bad, sizeof out, hipMemcpyDeviceToHost) == hipSuccess;
  }
  (void)hipFree(bad);
  std::printf("%llu %llu %llu\n", out[0], out[1], out[2]);
  return ok ? 0 : 1;
}
