// The steps of a small router as device functions, of the launch that takes them for a batch (front_kernel, moe_route.hip) and of the one
// that takes them in front of single tokens' experts (token_front_gateup_kernel, moe_token.hip): the bits of both hang on every
// operation and its place, so each stands here once.  Files that include this are compiled with -ffp-contract=off.
#pragma once
#include "moe_route_device.h"

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

// the squares of eight values, in their order
__device__ __forceinline__ float front_squares(const moe_bf16x8& in) {
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float v = bf16_to_f32(in.v[j]);
    ss = __fadd_rn(ss, __fmul_rn(v, v));
  }
  return ss;
}
// eight values normalised; total: the row's squares, wt: its norm's weights
__device__ __forceinline__ void front_norm(moe_bf16x8& in, float total, int D, float eps, const v4f (&wt)[2]) {
  const float rms = __fsqrt_rn(__fadd_rn(__fdiv_rn(total, (float)D), eps));
#pragma unroll
  for (int j = 0; j < 8; ++j) in.v[j] = f32_to_bf16(__fmul_rn(__fdiv_rn(bf16_to_f32(in.v[j]), rms), __fadd_rn(1.0f, wt[j / 4][j % 4])));
}
// a lane's part of a K block of the router's weights, up to GROUPS fragments of 16 columns; w: (E, D), extra: column E or null
template <int GROUPS>
__device__ __forceinline__ void front_weights(v4i (&b)[GROUPS][4], const bf16_t* w, const bf16_t* extra, int E, int N, int D, int block) {
  const int fr = threadIdx.x & 15, fq = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int g = 0; g < GROUPS; ++g) {
    if (16 * g >= N) break;
    const int n = min(16 * g + fr, N - 1);
    const v4i* src = (const v4i*)((n < E ? w + (size_t)n * D : extra) + block * 128) + fq;
#pragma unroll
    for (int s = 0; s < 4; ++s) b[g][s] = src[4 * s];
  }
}
// a K block's products of 16 rows with a fragment
__device__ __forceinline__ v4f front_products(const v4i (&rows)[4], const v4i (&b)[4]) {
  v4f acc = {};
#pragma unroll
  for (int s = 0; s < 4; ++s)
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, rows[s]), __builtin_bit_cast(bf16x8_t, b[s]), acc, 0, 0, 0);
  return acc;
}
// a column's logit from its blocks' products, `stride` apart
__device__ __forceinline__ float front_logit(const float* products, int KB, int stride) {
  float s = products[0];
  for (int kb = 1; kb < KB; ++kb) s = __fadd_rn(s, products[kb * stride]);
  return bf16_to_f32(f32_to_bf16(s));
}
__device__ __forceinline__ float front_gate(float logit) { return bf16_to_f32(f32_to_bf16(sigmoid_det(logit))); }
// eight values to codes; 16 lanes a quantisation group (moe_quant_act_block)
__device__ __forceinline__ uint2 front_codes(const moe_bf16x8& in, float& scale_inv) {
  float v[8], amax = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    v[j] = bf16_to_f32(in.v[j]);
    amax = fmaxf(amax, fabsf(v[j]));
  }
  unsigned m = __float_as_uint(amax);   // (not negative: ordered as integers)
  m = max(m, dpp<DPP_XOR1>(m));
  m = max(m, dpp<DPP_XOR2>(m));
  m = max(m, dpp<DPP_MIRROR8>(m));
  m = max(m, dpp<DPP_MIRROR16>(m));
  float scale;
  fp8_scales(__uint_as_float(m), scale, scale_inv);
  uint2 out;
  out.x = pack4_e4m3(v[0] * scale, v[1] * scale, v[2] * scale, v[3] * scale);
  out.y = pack4_e4m3(v[4] * scale, v[5] * scale, v[6] * scale, v[7] * scale);
  return out;
}

}  // namespace
