// Status reporting of the C ABI: the reason for the calling thread's last non-OK status.
#include <algorithm>
#include <cstdio>

#include "common.h"

namespace ishz {
static thread_local std::string t_last_error;

void set_error(const std::string &msg) { t_last_error = msg; }

int fail(const char *what, hipError_t e) {
  set_error(std::string(what) + ": " + hipGetErrorString(e));
  return ISHZ_EHIP;
}

int decline(const std::string &why) {
  set_error("declined: " + why);
  return ISHZ_DECLINED;
}

int einval(const std::string &why) {
  set_error("invalid argument: " + why);
  return ISHZ_EINVAL;
}

// One workgroup per row: the row's largest magnitude, then every value times 2^-e rounded to fp16.
// A row is a few tens of KB, so latency bounds it: every thread has its whole share of the row (up
// to U 16-byte loads) in flight at once and keeps it in registers between the two passes. With one
// 2-byte load per value and 256 threads, K = 5120 took 10 us and K = 25600 60 us.
__global__ __launch_bounds__(1024) void act_half_kernel(const uint16_t *__restrict__ x, int K,
                                                        uint16_t *__restrict__ xh, float *__restrict__ rs) {
  __shared__ uint32_t wmax[16];
  constexpr int U = 4;  // 1024 threads hold 32768 values; longer rows are read again by the second pass
  const int n8 = K / 8, nt = blockDim.x;
  const u4 *src = (const u4 *)(x + (size_t)blockIdx.x * K);
  u4 *dst = (u4 *)(xh + (size_t)blockIdx.x * K);
  u4 v[U];
  auto load = [&](int i0) {
#pragma unroll
    for (int u = 0; u < U; u++) v[u] = ld16<2>((const uint8_t *)(src + min(i0 + u * nt, n8 - 1)));
  };
  uint32_t m = 0;
  for (int i0 = threadIdx.x; i0 < n8; i0 += U * nt) {
    load(i0);
#pragma unroll
    for (int u = 0; u < U; u++) m = bf16_absmax(v[u], m);
  }
  const int e = bf16_row_exponent(block_absmax(m, wmax));
  const float down = ldexpf(1.0f, -e);
  for (int i0 = threadIdx.x; i0 < n8; i0 += U * nt) {
    if (n8 > U * nt) load(i0);
#pragma unroll
    for (int u = 0; u < U; u++)
      if (i0 + u * nt < n8) dst[i0 + u * nt] = bf16_to_half8(v[u], down);
  }
  if (threadIdx.x == 0) rs[blockIdx.x] = ldexpf(1.0f, e);
}

size_t act_image_bytes(int M, int K) { return ((size_t)M * K * 2 + 255) / 256 * 256 + ((size_t)M * 4 + 255) / 256 * 256; }

int act_prepare(const void *x, int dt, int M, int K, void *image, hipStream_t st, const uint16_t **xh,
                const float **rs) {
  if (dt == ISHZ_DT_F16) {
    *xh = (const uint16_t *)x;
    *rs = nullptr;
    return ISHZ_OK;
  }
  if (dt != ISHZ_DT_BF16 || K % 8) return decline("the fp16 image takes bf16 rows of a multiple of 8 values");
  if (!image) return einval("bf16 activations need a workspace");
  uint16_t *h = (uint16_t *)image;
  float *r = (float *)((char *)image + ((size_t)M * K * 2 + 255) / 256 * 256);
  const int nt = std::min(1024, (K / 8 + 63) / 64 * 64);
  hipLaunchKernelGGL(act_half_kernel, dim3(M), dim3(nt), 0, st, (const uint16_t *)x, K, h, r);
  ISHZ_LAUNCH_CHECK("activation image launch");
  *xh = h;
  *rs = r;
  return ISHZ_OK;
}
}  // namespace ishz

extern "C" const char *ishz_last_error(void) { return ishz::t_last_error.c_str(); }
extern "C" int ishz_version(void) { return 100; }
