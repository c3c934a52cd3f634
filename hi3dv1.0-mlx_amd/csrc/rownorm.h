// fp16 row-normalisation steps shared by the LayerNorm kernels (norm.hip) and the
// convolution epilogues that apply the res block's second norm (conv.hip, conv_group.hip).
//
// Reference: layer_norm_modulate (src/hi3d_mac/mlx_backend/kernels.py:162-237) and the
// fp16 SiLU of the res blocks (src/hi3d_mac/mlx_backend/transformer.py:172-173).
#pragma once

#include "conv_tile.h"
#include "quant.h"

namespace hi3d {

// SiLU of an fp16 value as the reference's fp16 ``x * sigmoid(x)``
// (src/hi3d_mac/mlx_backend/transformer.py:172-173): the sigmoid rounded to fp16, then
// the product rounded to fp16. The sigmoid runs through the hardware exp2 and
// reciprocal (~1 ulp each in fp32); its fp16 rounding differs from that of the exact
// sigmoid in about one value in 10^4. The product of two fp16 values is exact in fp32,
// so the native fp16 multiply rounds it as the fp32 product rounded to fp16 does.
__device__ __forceinline__ _Float16 silu_h(_Float16 h) {
#pragma clang fp contract(off)
  const float x = static_cast<float>(h);
  const _Float16 sig = static_cast<_Float16>(__builtin_amdgcn_rcpf(1.0f + __expf(-x)));
  return h * sig;
}

// The norm's f32 value, rounded to f32 and kept as such before its conversion to fp16:
// without this the compiler folds fp16((x - mean) * inv) into one mixed-precision FMA
// (v_fma_mixlo_f16), which rounds the exact product to fp16 once instead of to f32 and
// then to fp16, and differs from the reference in rare last bits.
__device__ __forceinline__ float f32_rounded(float y) {
  asm("" : "+v"(y));
  return y;
}

// fp16(fp16(h * scale) + shift) on 8 columns with native fp16 multiplies and adds (no
// FMA). The reference rounds each step through fp32; a product of two fp16 values is
// exact in fp32, and fp32 carries more than twice fp16's precision plus two bits, so
// rounding through fp32 and rounding once give the same fp16 results.
__device__ __forceinline__ f16x8 modulate8(f16x8 h, f16x8 scale, f16x8 shift) {
#pragma clang fp contract(off)
  const f16x8 p = h * scale;
  return p + shift;
}

// The res block's second norm on a 128-channel row held by eight lanes (lane % 8 = g has
// chunks g and g + 8): LayerNorm, the modulation and SiLU with the lanes, chunks,
// summation order and reduction partners of ln_kernel<8, 2> (by DPP moves), so that a
// convolution that ends with it gives the bits of the convolution followed by that kernel.
__device__ __forceinline__ void ln_modulate_silu_row128(f16x8 (&h)[2], float eps, const _Float16* scale,
                                                        const _Float16* shift, int g) {
#pragma clang fp contract(off)
  const float c = 128.0f;
  float v[2][8];
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[i][e] = static_cast<float>(h[i][e]);
      sum += v[i][e];
    }
  sum += dpp_xor4(sum);
  sum += dpp_xor2(sum);
  sum += dpp_xor1(sum);
  const float mean = sum / c;
  float sq = 0.0f;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float d = v[i][e] - mean;
      sq += d * d;
    }
  sq += dpp_xor4(sq);
  sq += dpp_xor2(sq);
  sq += dpp_xor1(sq);
  const float inv = 1.0f / sqrtf(sq / c + eps);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int ch = (g + 8 * i) * 8;
#pragma unroll
    for (int e = 0; e < 8; ++e) h[i][e] = static_cast<_Float16>(f32_rounded((v[i][e] - mean) * inv));
    h[i] = modulate8(h[i], *reinterpret_cast<const f16x8*>(scale + ch), *reinterpret_cast<const f16x8*>(shift + ch));
#pragma unroll
    for (int e = 0; e < 8; ++e) h[i][e] = silu_h(h[i][e]);
  }
}

}  // namespace hi3d
