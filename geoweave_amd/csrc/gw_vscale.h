// The fp16 scaling of V shared by the masked dense and the union forward.
#pragma once

#include <math.h>

#include "gw_dense.h"

namespace gw {
namespace {

// ---------------------------------------------------------------------------------------
// V enters the P·V product in fp16, scaled per (head, d) column by a power of two 2^e that
// puts the column's largest |v| in [2^14, 2^15): the scaling is exact, every scaled value
// fits fp16, and values down to 2^-28 of the column's largest stay normal. o is scaled back
// by 2^-e. dense_vmax_kernel takes the column maxima (as ordered bit patterns of
// non-negative floats, atomic max); columns that are all zero or hold inf/nan keep e = 0.
// It reads the K rows of the same keys and head too, and sets bad[b] when any K or V value
// of the batch element is an inf or a nan (exponent field all ones).
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ int vscale_exp(uint32_t bits) {
  const float mx = __uint_as_float(bits);
  if (!(mx > 0.f) || !(mx <= 3.4028234663852886e38f)) return 0;
  int x;
  frexpf(mx, &x);  // mx = f 2^x, f in [0.5, 1)
  return min(15 - x, 126);
}

constexpr int kVmaxKeys = 256;  // keys per workgroup of dense_vmax_kernel (one head)

__global__ __launch_bounds__(256) void dense_vmax_kernel(const uint16_t* __restrict__ v, int64_t vsb, int64_t vss,
                                                         int64_t vsh, const uint16_t* __restrict__ k, int64_t ksb,
                                                         int64_t kss, int64_t ksh, int S, int H, int in_fp16,
                                                         uint32_t* __restrict__ vmax, int* __restrict__ bad) {
  __shared__ float part[4][64];
  const int h = blockIdx.y, b = blockIdx.z;
  const int dc = threadIdx.x & 7, kr = threadIdx.x >> 3;  // 16-byte chunk of the row, key
  const int s0 = blockIdx.x * kVmaxKeys;
  const uint16_t* src = v + b * vsb + h * vsh + dc * 8;
  const uint16_t* ksrc = k + b * ksb + h * ksh + dc * 8;
  const uint32_t e = in_fp16 ? 0x7C00u : 0x7F80u;
  float mx[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) mx[i] = 0.f;
  uint4 val[8], kval[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const int s = s0 + kr + 32 * u;
    val[u] = s < S ? *reinterpret_cast<const uint4*>(src + (int64_t)s * vss) : make_uint4(0, 0, 0, 0);
    kval[u] = s < S ? *reinterpret_cast<const uint4*>(ksrc + (int64_t)s * kss) : make_uint4(0, 0, 0, 0);
  }
  uint32_t nf = 0u;
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const uint32_t w[4] = {val[u].x, val[u].y, val[u].z, val[u].w};
    const uint32_t kw[4] = {kval[u].x, kval[u].y, kval[u].z, kval[u].w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      mx[2 * i] = fmaxf(mx[2 * i], fabsf(in_to_float(in_fp16, w[i] & 0xFFFFu)));
      mx[2 * i + 1] = fmaxf(mx[2 * i + 1], fabsf(in_to_float(in_fp16, w[i] >> 16)));
      nf |= nonfinite2(w[i], e) | nonfinite2(kw[i], e);
    }
  }
  if (nf != 0u) bad[b] = 1;  // every writer stores the same value
  // lanes with the same chunk: xor 8, 16, 32; then the four waves
#pragma unroll
  for (int i = 0; i < 8; ++i) {
#pragma unroll
    for (int off = 8; off < 64; off <<= 1) mx[i] = fmaxf(mx[i], __shfl_xor(mx[i], off));
  }
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane < 8) {
#pragma unroll
    for (int i = 0; i < 8; ++i) part[wave][lane * 8 + i] = mx[i];
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    const float m4 = fmaxf(fmaxf(part[0][threadIdx.x], part[1][threadIdx.x]), fmaxf(part[2][threadIdx.x], part[3][threadIdx.x]));
    atomicMax(vmax + ((int64_t)b * H + h) * 64 + threadIdx.x, __float_as_uint(m4));
  }
}

}  // namespace
}  // namespace gw
