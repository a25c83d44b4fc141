// Block-scaled e4m3fn quantisers (HBM-bound, 16-byte accesses).
//
// scale = 448/amax, q = e4m3(clamp(x*scale, +-448)), stored scale = 1/scale.
// Activations: 1x128 groups (replaces the per-row quantiser of
// jax_gpt/models/qwen35/fp8.py:30-45).  Weights: 128x128 blocks in the
// (E, out, in) layout of quantize.py:31-42.
#include "moe_common.h"
#include "moe_quant_device.h"

namespace {

typedef moe_bf16x8 bf16x8;

__global__ __launch_bounds__(256) void quant_act_kernel(const QuantJob q) { moe_quant_act_block(q, blockIdx.x); }

// RMSNorm fused with the activation quantiser: one workgroup per row, thread t holds the row's 16-byte piece t between
// the two passes, so that the 16 lanes of a quantisation group are neighbours as in quant_act_kernel.
// normed = bf16((x / sqrt(mean(x^2) + eps)) * (1 + weight)), the Qwen3.5 convention of
// jax_gpt/models/qwen35/primitives.py:16-32 (the step in front of the MoE layer, block.py:54 and :88), then
// the 1x128 quantisation of the bf16 values.  Sums are taken in a fixed order with individually rounded operations: the
// first 256 threads add the squares of pieces t, t + 256, ... (through LDS where there are several).
//   A launch of few rows is bound by latency, and straight-line code is part of it: some 0.3 us per KB that the first
// wave has to fetch.  With four pieces per thread whatever D is (12.7 KB) and the weights read behind the sum 1 row of
// 1024 took 6.3 us and 32 rows of 4096 9.7; this way
// 2.6 and 5.0 (4096 rows of 4096: 51 and 25 us).
constexpr int kNormPieces = 4;   // D <= 256 * 8 * 4 = 8192

template <int PIECES>
__global__ __launch_bounds__(256 * PIECES) void rmsnorm_quant_kernel(const void* __restrict__ x, int x_f32,
                                                                    const float* __restrict__ weight, float eps, int D,
                                                                    bf16x8* __restrict__ normed, uint2* __restrict__ xq,
                                                                    float* __restrict__ sx, float* __restrict__ sx_blocked) {
  __shared__ float wave_sum[4];
  __shared__ v4i raw[PIECES > 1 ? 256 * PIECES : 1];
  const int row = blockIdx.x, P = D / 8, t = threadIdx.x;
  const bool ok = t < P;              // uniform over the 16 lanes of a group (P is a multiple of 16)
  bf16x8 in = {};
  float wt[8] = {};
  if (ok) {
    in = load_bf16x8(x, x_f32, (size_t)row * P + t);
#pragma unroll
    for (int j = 0; j < 8; ++j) wt[j] = weight[t * 8 + j];
  }
  if (PIECES > 1) {
    raw[t] = __builtin_bit_cast(v4i, in);
    __syncthreads();
  }
  if (t < 256) {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const bf16x8 v = i == 0 ? in : __builtin_bit_cast(bf16x8, raw[t + 256 * i]);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float f = bf16_to_f32(v.v[j]);
        ss = __fadd_rn(ss, __fmul_rn(f, f));
      }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) ss = __fadd_rn(ss, __shfl_xor(ss, off, MOE_WAVE));
    if ((t & 63) == 0) wave_sum[t >> 6] = ss;
  }
  __syncthreads();
  if (!ok) return;
  const float total = __fadd_rn(__fadd_rn(wave_sum[0], wave_sum[1]), __fadd_rn(wave_sum[2], wave_sum[3]));
  const float rms = __fsqrt_rn(__fadd_rn(__fdiv_rn(total, (float)D), eps));
  float f[8], amax = 0.f;
  bf16x8 nb;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    nb.v[j] = f32_to_bf16(__fmul_rn(__fdiv_rn(bf16_to_f32(in.v[j]), rms), __fadd_rn(1.0f, wt[j])));
    f[j] = bf16_to_f32(nb.v[j]);
    amax = fmaxf(amax, fabsf(f[j]));
  }
#pragma unroll
  for (int off = 1; off < 16; off <<= 1) amax = fmaxf(amax, __shfl_xor(amax, off, MOE_WAVE));
  float scale, scale_inv;
  fp8_scales(amax, scale, scale_inv);
  const size_t at = (size_t)row * P + t;
  if (normed) normed[at] = nb;
  uint2 out;
  out.x = pack4_e4m3(f[0] * scale, f[1] * scale, f[2] * scale, f[3] * scale);
  out.y = pack4_e4m3(f[4] * scale, f[5] * scale, f[6] * scale, f[7] * scale);
  xq[at] = out;
  if ((t & 15) == 0) {
    sx[at >> 4] = scale_inv;
    if (sx_blocked) sx_blocked[(size_t)(t >> 4) * gridDim.x + row] = scale_inv;   // the (K/128, M) array
  }
}

// One workgroup per 128x128 block, or for two of them side by side (WIDE).  A lane takes 16 bytes of a row (8 bf16 or 4 f32), 16 or
// 32 neighbouring lanes a block's row, so a wave's loads and stores are whole lines; the blocks stay in registers, packed,
// between the maximum and the rounding.  HBM-bound: every byte is read once and written once, hence non-temporal.  16 x 2048 x 7168
// bf16: 158 us as 64 consecutive elements per thread, 118 us as a block a workgroup of four waves (5.97 TB/s; without the hints 130
// us), 111 as two of sixteen (6.3); f32 191 and, with sixteen waves, 182 (6.5).  Which form where: moe_quant_weight_block.
template <typename T, int WIDE, int THREADS>
__global__ __launch_bounds__(THREADS) void quant_weight_kernel(const T* __restrict__ w, int N, int K,
                                                              uint8_t* __restrict__ wq, float* __restrict__ sw) {
  constexpr int V = 16 / sizeof(T), kBlockLanes = 128 / V, kRowLanes = WIDE * kBlockLanes, kStepRows = THREADS / kRowLanes, kSteps = 128 / kStepRows;
  __shared__ float red[kStepRows][WIDE];
  const int nb = blockIdx.y, e = blockIdx.z;
  const int row0 = threadIdx.x / kRowLanes, lane = threadIdx.x % kRowLanes, block = lane / kBlockLanes, kb = blockIdx.x * WIDE + block;
  const size_t off = ((size_t)e * N + (size_t)nb * 128 + row0) * K + (size_t)blockIdx.x * (WIDE * 128) + lane * V;
  const size_t step = (size_t)kStepRows * K;
  v4i raw[kSteps];
#pragma unroll
  for (int i = 0; i < kSteps; ++i) raw[i] = __builtin_nontemporal_load((const v4i*)(w + off + i * step));
  auto value = [&](int i, int j) {   // j-th of the lane's values of step i
    if constexpr (V == 4) return __int_as_float(raw[i][j]);
    else return __int_as_float((j & 1) ? (raw[i][j >> 1] & 0xffff0000) : (raw[i][j >> 1] << 16));
  };
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < kSteps; ++i)
#pragma unroll
    for (int j = 0; j < V; ++j) amax = fmaxf(amax, fabsf(value(i, j)));
#pragma unroll
  for (int o = kBlockLanes / 2; o >= 1; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, MOE_WAVE));
  if (lane % kBlockLanes == 0) red[row0][block] = amax;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kStepRows; ++i) amax = fmaxf(amax, red[i][block]);
  float scale, scale_inv;
  fp8_scales(amax, scale, scale_inv);
#pragma unroll
  for (int i = 0; i < kSteps; ++i) {
    typedef unsigned codes_t __attribute__((ext_vector_type(V / 4)));
    codes_t out;
#pragma unroll
    for (int q = 0; q < V / 4; ++q)
      out[q] = pack4_e4m3(value(i, 4 * q) * scale, value(i, 4 * q + 1) * scale, value(i, 4 * q + 2) * scale, value(i, 4 * q + 3) * scale);
    __builtin_nontemporal_store(out, (codes_t*)(wq + off + i * step));
  }
  if (row0 == 0 && lane % kBlockLanes == 0) sw[((size_t)e * (N / 128) + nb) * (K / 128) + kb] = scale_inv;
}

}  // namespace

extern "C" int moe_quant_act(const void* x_bf16, int R, int K, uint8_t* xq, float* sx, moe_stream_t stream) {
  return moe_quant_act_impl(x_bf16, 0, nullptr, R, K, xq, sx, nullptr, stream);
}
// checks the arguments of an activation quantisation and describes it (for its own launch, or a routing launch's)
int moe_quant_act_job(const void* x, int x_f32, void* x_bf16, int R, int K, uint8_t* xq, float* sx, float* sx_blocked, QuantJob* job) {
  MOE_REQUIRE(R == 0 || (x && xq && sx), MOE_ERR_NULL, "quant_act: null pointer");
  MOE_REQUIRE(R >= 0 && K > 0 && K % MOE_QBLOCK == 0, MOE_ERR_BAD_SHAPE, "quant_act: K=%d must be a positive multiple of 128 (R=%d)", K, R);
  MOE_REQUIRE(MOE_ALIGNED16(x) && MOE_ALIGNED16(xq), MOE_ERR_BAD_ALIGN, "quant_act: pointers must be 16-byte aligned");
  const long long pieces = (long long)R * K / 8;
  MOE_REQUIRE(pieces < (1ll << 38), MOE_ERR_BAD_SHAPE, "quant_act: too many elements");
  *job = QuantJob{x, x_f32, x_bf16, pieces, K / 128, R, xq, sx, sx_blocked};
  return MOE_OK;
}
int moe_quant_act_impl(const void* x, int x_f32, void* x_bf16, int R, int K, uint8_t* xq, float* sx, float* sx_blocked,
                       moe_stream_t stream) {
  QuantJob job;
  if (int rc = moe_quant_act_job(x, x_f32, x_bf16, R, K, xq, sx, sx_blocked, &job)) return rc;
  if (R == 0) return MOE_OK;
  hipLaunchKernelGGL(quant_act_kernel, dim3(moe_quant_blocks(job, 256)), dim3(256), 0, (hipStream_t)stream, job);
  return moe_check_hip(hipGetLastError(), "quant_act launch");
}

extern "C" int moe_rmsnorm_quant(const void* x_bf16, const float* weight, float eps, int M, int D, void* normed_bf16,
                                 uint8_t* xq, float* sx, moe_stream_t stream) {
  return moe_rmsnorm_quant_impl(x_bf16, 0, weight, eps, M, D, normed_bf16, xq, sx, nullptr, stream);
}
int moe_rmsnorm_quant_impl(const void* x, int x_f32, const float* weight, float eps, int M, int D, void* normed_bf16,
                           uint8_t* xq, float* sx, float* sx_blocked, moe_stream_t stream) {
  MOE_REQUIRE((M == 0 || (x && xq && sx)) && weight, MOE_ERR_NULL, "rmsnorm_quant: null pointer");
  MOE_REQUIRE(M >= 0 && D > 0 && D % MOE_QBLOCK == 0 && D <= 256 * 8 * kNormPieces, MOE_ERR_BAD_SHAPE,
              "rmsnorm_quant: D=%d must be a multiple of 128, at most %d (M=%d)", D, 256 * 8 * kNormPieces, M);
  MOE_REQUIRE(MOE_ALIGNED16(x) && MOE_ALIGNED16(xq) && MOE_ALIGNED16(normed_bf16), MOE_ERR_BAD_ALIGN,
              "rmsnorm_quant: pointers must be 16-byte aligned");
  if (M == 0) return MOE_OK;
  auto launch = [&](auto* kernel, int pieces) {
    hipLaunchKernelGGL(kernel, dim3(M), dim3(256 * pieces), 0, (hipStream_t)stream, x, x_f32, weight, eps, D,
                       (bf16x8*)normed_bf16, (uint2*)xq, sx, sx_blocked);
  };
  if (D <= 2048) launch(rmsnorm_quant_kernel<1>, 1);
  else if (D <= 4096) launch(rmsnorm_quant_kernel<2>, 2);
  else launch(rmsnorm_quant_kernel<kNormPieces>, kNormPieces);
  return moe_check_hip(hipGetLastError(), "rmsnorm_quant launch");
}

extern "C" int moe_quant_weight_block(const void* w, int src_is_f32, int E, int N, int K, uint8_t* wq,
                                      float* sw, moe_stream_t stream) {
  MOE_REQUIRE(w && wq && sw, MOE_ERR_NULL, "quant_weight_block: null pointer");
  MOE_REQUIRE(E >= 1 && N > 0 && K > 0 && N % 128 == 0 && K % 128 == 0 && E < 65536 && N / 128 < 65536,
              MOE_ERR_BAD_SHAPE, "quant_weight_block: N=%d and K=%d must be multiples of 128 (E=%d)", N, K, E);
  MOE_REQUIRE(MOE_ALIGNED16(w) && MOE_ALIGNED16(wq), MOE_ERR_BAD_ALIGN, "quant_weight_block: pointers must be 16-byte aligned");
  // Large arrays take workgroups of sixteen waves, bf16 two blocks wide: 512 bytes of a row, as f32 rows are with one.  Weights and
  // codes together in MB, us with one block and four waves / this way, other weights and codes each time:
  //   bf16 96 18.9 / 19.1, 129 24.7 / 25.3, 144 26.8 / 27.1, 185 33.7 / 33.3, 208 36.1 / 35.3, 270 48.0 / 47.7, 336 58.9 / 56.4, 562
  // 98.8 / 93.2, 672 119.2 / 111.4, 2352 429 / 389;
  //   f32 160 29.3 / 30.8, 216 37.8 / 37.3, 320 56.6 / 56.9, 347 60.0 / 56.9, 450 75.4 / 74.8, 560 94.9 / 89.8, 957 167 / 154, 1120 191 / 182.
  // Below, f32 takes eight waves, or four where a CU has between one and two blocks (blocks of 128 x 128, us with four / eight): 256 5.69 /
  // 5.49, 320 7.07 / 6.87, 384 7.54 / 7.63, 440 7.85 / 8.09, 500 8.47 / 8.77, 520 10.45 / 10.26, 576 10.59 / 10.26, 768 12.60 / 12.36, 896
  // 13.99 / 14.19, 1024 16.06 / 15.66, 1536 22.32 / 22.50, 2560 36.0 / 35.9.  Plain stores look 9 % better only while the same codes are written again and
  // again and stay in the memory-side cache (672 MB: 107; into other memory each time 123).
  const long long n = (long long)E * N * K;
  auto launch = [&](auto* kernel, auto* src, int width, int threads) {
    hipLaunchKernelGGL(kernel, dim3(K / (128 * width), N / 128, E), dim3(threads), 0, (hipStream_t)stream, src, N, K, wq, sw);
  };
  const long long blocks = n / (128 * 128);
  if (src_is_f32) n * 5 > (320ll << 20) ? launch(quant_weight_kernel<float, 1, 1024>, (const float*)w, 1, 1024)
                  : blocks > 320 && blocks <= 512 ? launch(quant_weight_kernel<float, 1, 256>, (const float*)w, 1, 256)
                                                  : launch(quant_weight_kernel<float, 1, 512>, (const float*)w, 1, 512);
  else n * 3 > (160ll << 20) && K % 256 == 0 ? launch(quant_weight_kernel<bf16_t, 2, 1024>, (const bf16_t*)w, 2, 1024)
                                             : launch(quant_weight_kernel<bf16_t, 1, 256>, (const bf16_t*)w, 1, 256);
  return moe_check_hip(hipGetLastError(), "quant_weight_block launch");
}

namespace {
// f32 <-> bf16 conversion of a flat array (the layer computes from bf16 activations and returns its caller's
// dtype, moe.py:282): round-to-nearest-even one way, exact the other
__global__ __launch_bounds__(256) void convert_kernel(const void* __restrict__ src, int src_is_f32, void* __restrict__ dst,
                                                     int dst_is_f32, long long n) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float v = src_is_f32 ? ((const float*)src)[i] : bf16_to_f32(((const bf16_t*)src)[i]);
  if (dst_is_f32) ((float*)dst)[i] = v;
  else ((bf16_t*)dst)[i] = f32_to_bf16(v);
}
}  // namespace

extern "C" int moe_convert(const void* src, int src_is_f32, void* dst, int dst_is_f32, long long n, moe_stream_t stream) {
  MOE_REQUIRE(n >= 0 && n < (1ll << 38), MOE_ERR_BAD_SHAPE, "convert: bad element count %lld", n);
  MOE_REQUIRE(n == 0 || (src && dst), MOE_ERR_NULL, "convert: null pointer");
  if (n == 0) return MOE_OK;
  hipLaunchKernelGGL(convert_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, src, src_is_f32,
                     dst, dst_is_f32, n);
  return moe_check_hip(hipGetLastError(), "convert launch");
}

namespace {
// Activation scales, row-major (rows, KB) -> block-major (KB, n) in row-list order: out[kb][p] = sx[ids ? ids[p] : p][kb].
// A thread takes kGatherScales neighbouring scales of one list position (half a line) and writes one float into each of as
// many output rows, where neighbouring threads write neighbouring floats.  Bound by latency (7 MB for 16384 rows of 56): with
// all scales of a row in one thread, 64 workgroups of 14 loads a thread, that took 8.2 us, now 4.5; 6216 rows of 56 6.4 -> 4.1.
constexpr int kGatherScales = 16;
__global__ __launch_bounds__(256) void gather_scales_kernel(const float* __restrict__ sx, const int32_t* __restrict__ ids,
                                                           int n, int KB, float* __restrict__ out) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= n) return;
  const float* row = sx + (size_t)(ids ? ids[p] : p) * KB;
  out += p;
  for (int kb0 = blockIdx.y * kGatherScales; kb0 < KB; kb0 += gridDim.y * kGatherScales) {
    const int m = min(kGatherScales, KB - kb0);
    if ((KB & 3) == 0) {
      float4 v[kGatherScales / 4];
#pragma unroll
      for (int i = 0; i < kGatherScales; i += 4)
        if (i < m) v[i / 4] = *(const float4*)(row + kb0 + i);
#pragma unroll
      for (int i = 0; i < kGatherScales; i += 4) {
        if (i >= m) break;
        float* o = out + (size_t)(kb0 + i) * n;
        o[0] = v[i / 4].x;
        o[(size_t)n] = v[i / 4].y;
        o[(size_t)2 * n] = v[i / 4].z;
        o[(size_t)3 * n] = v[i / 4].w;
      }
    } else {
      for (int i = kb0; i < kb0 + m; ++i) out[(size_t)i * n] = row[i];
    }
  }
}
}  // namespace

extern "C" int moe_gather_scales(const float* sx, const int32_t* row_ids, int n, int KB, float* out, moe_stream_t stream) {
  MOE_REQUIRE(n >= 0 && KB >= 1, MOE_ERR_BAD_SHAPE, "gather_scales: bad sizes n=%d KB=%d", n, KB);
  MOE_REQUIRE(n == 0 || (sx && out), MOE_ERR_NULL, "gather_scales: null pointer");
  // (rows of a multiple of four scales are read 16 bytes at a time)
  MOE_REQUIRE((KB & 3) || MOE_ALIGNED16(sx), MOE_ERR_BAD_ALIGN, "gather_scales: sx must be 16-byte aligned when KB is a multiple of 4");
  if (n == 0) return MOE_OK;
  const int parts = KB / kGatherScales + (KB % kGatherScales ? 1 : 0);
  hipLaunchKernelGGL(gather_scales_kernel, dim3((unsigned)((n + 255) / 256), parts < 64 ? parts : 64), dim3(256), 0, (hipStream_t)stream, sx, row_ids,
                     n, KB, out);
  return moe_check_hip(hipGetLastError(), "gather_scales launch");
}
