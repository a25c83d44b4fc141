// Routing: one wavefront per token, and with it the rest of what stands in front of the grouped GEMMs.
//
// Selection is exact integer work on order-preserving keys, so the indices do
// not depend on any transcendental: softmax routing ranks the logits (softmax
// is monotone), and the group-limited sigmoid router ranks sigmoid(logit)+bias
// where sigmoid is computed by a fixed sequence of individually rounded f32
// operations (no fused multiply-add; this file is compiled with
// -ffp-contract=off) that a CPU can repeat bit for bit.
//
// Replaces jax_gpt/models/qwen35/moe.py:51-53 (softmax, lax.top_k, renormalise) and, for a whole layer, the
// counting half of :58-80.
#include "moe_common.h"
#include "moe_permute_device.h"
#include "moe_quant_device.h"
#include "moe_front_device.h"

namespace {

// Columns [0, n) of the partial sums at p, added in slice order by the whole workgroup and rounded to bf16 (what the
// router's own finishing pass computes).  The loads are what it waits for, so a thread has up to 8 slices of C columns
// under way: past the last slice or column it reads the last one again.  (One column and batches of 8, 4, 1, 1, ...: the
// launch took 24 us for 2047 tokens of 513 columns in 7 slices, 20 now.  Sixteen slices of one column: 9.2 against 9.3 us for
// 1 token of 32 slices, and the code alone costs 0.7 us where there are few: mini layer, 3000 tokens 5.2 -> 6.0.)
template <int Z, int C>
__device__ __forceinline__ void add_slices(float (&s)[C], const float* const (&q)[C], size_t slice, int z, int splits) {
  float v[Z][C];
#pragma unroll
  for (int j = 0; j < Z; ++j)
#pragma unroll
    for (int c = 0; c < C; ++c) v[j][c] = q[c][(size_t)min(z + j, splits - 1) * slice];
#pragma unroll
  for (int j = 0; j < Z; ++j)
#pragma unroll
    for (int c = 0; c < C; ++c) s[c] = z + j == 0 ? v[j][c] : z + j < splits ? __fadd_rn(s[c], v[j][c]) : s[c];
}
template <int C>
__device__ __forceinline__ void sum_partials(const float* p, size_t slice, int splits, int n, float* rows) {
  for (int i0 = threadIdx.x; i0 < n; i0 += C * blockDim.x) {
    float s[C] = {};
    const float* q[C];
#pragma unroll
    for (int c = 0; c < C; ++c) q[c] = p + min(i0 + c * (int)blockDim.x, n - 1);
    int z = 0;
    for (; splits - z > 4; z += 8) add_slices<8, C>(s, q, slice, z, splits);
    if (splits - z > 1) add_slices<4, C>(s, q, slice, z, splits);
    else if (splits - z == 1) add_slices<1, C>(s, q, slice, z, splits);
#pragma unroll
    for (int c = 0; c < C; ++c)
      if (i0 + c * (int)blockDim.x < n) rows[i0 + c * (int)blockDim.x] = bf16_to_f32(f32_to_bf16(s[c]));
  }
}

// Workgroup c routes tokens [c * tokens_per_block, +tokens_per_block).  Around the selection:
//  - LogitSource's partial sums are added by the whole workgroup for as many tokens as it has waves (a token's columns
//    are contiguous in every slice: independent coalesced loads, see sum_partials) and the waves then read the rounded
//    logits from LDS.  One wave summing its own token one load at a time took 87 us for 32 tokens of 513 columns in
//    32 slices, most of the layer's overhead; this way 9 us.
//  - chunk_hist: the workgroup's selections are counted for the sort by expert (one row of E counts per workgroup;
//    not where so few rows would leave CUs idle, see moe_route_impl).
//  - sort_here (one workgroup routes the whole batch): the sort itself follows in the same launch.
//  - the blocks behind the routing blocks quantise the activations: independent work, one launch less.
struct RouteJob {
  int blocks, tokens_per_block, batch;   // batch: tokens whose partial sums are added at a time
  int32_t* chunk_hist;                   // [blocks][E] or null
};
// A batch that one workgroup routes and sorts (16 waves, a token each at a time) against a second launch for the sort:
// 12 tokens of the tiny layer 26 / 22 us, 32 of it 26.0 / 24.9, 48 25.9 / 26.6; 12 and 16 of the mini layer 36.5 / 35;
// 12 of the DeepSeek-V3 layer (96 entries) 379.1 / 379.8, 32 of the Qwen3-MoE layer (256 entries) 103.3 / 105.9.
inline bool route_sorts_here(int M, int k, bool partial) { return M <= 8 || (M * k <= 64 && M <= (partial ? 16 : 32)); }

template <int VPL, int KIND, bool SORT_HERE>
__global__ __launch_bounds__(1024) void route_kernel(const RouteArgs a, const RouteJob job, const QuantJob quant, const PermuteOut sort) {
  if ((int)blockIdx.x >= job.blocks) {
    moe_quant_act_block(quant, (int)blockIdx.x - job.blocks);
    return;
  }
  extern __shared__ __attribute__((aligned(16))) int lds[];   // [ids when sort_here][E counts][logits or the sort's counters]
  int* ids = lds;
  int* hist = lds + (SORT_HERE ? kSmallRows : 0);
  float* rows = (float*)(hist + a.E);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const int first = blockIdx.x * job.tokens_per_block, last = min(a.M, first + job.tokens_per_block);
  if (!SORT_HERE && job.chunk_hist)
    for (int e = threadIdx.x; e < a.E; e += blockDim.x) hist[e] = 0;
  __syncthreads();
  const int N = a.src.N;
  for (int t0 = first; t0 < last; t0 += job.batch) {
    const int nt = min(job.batch, last - t0);
    if (a.src.partial) {
      if (t0 > first) __syncthreads();   // (the waves are done with the batch before)
      const size_t MN = (size_t)a.M * N;
      const float* p = a.src.partial + (size_t)t0 * N;
      if (nt * N > (int)blockDim.x) sum_partials<2>(p, MN, a.src.splits, nt * N, rows);
      else sum_partials<1>(p, MN, a.src.splits, nt * N, rows);
      __syncthreads();
    }
    for (int tt = wave; tt < nt; tt += waves) {
      const int t = t0 + tt;
      const float* row = a.src.partial ? rows + tt * N : a.src.logits + (size_t)t * a.E;
      if (a.src.partial) {
        if (a.src.out_logits)
          for (int e = lane; e < a.E; e += MOE_WAVE) a.src.out_logits[(size_t)t * a.E + e] = row[e];
        if (lane == 0 && a.src.shared_gate && N > a.E)   // the shared expert's gate rides in column E
          a.src.shared_gate[t] = front_gate(row[a.E]);
      }
      const int chosen = KIND == ROUTE_SOFTMAX ? route_softmax_token<VPL>(a, row, t).expert : route_grouped_token<VPL>(a, row, t).expert;
      if (lane < a.k) {
        if (!SORT_HERE && job.chunk_hist) atomicAdd(&hist[chosen], 1);
        if (SORT_HERE) ids[t * a.k + lane] = chosen;
      }
    }
  }
  if (!SORT_HERE && job.chunk_hist) {
    __syncthreads();
    for (int e = threadIdx.x; e < a.E; e += blockDim.x) job.chunk_hist[(size_t)blockIdx.x * a.E + e] = hist[e];
  }
  if (SORT_HERE) {
    __syncthreads();
    permute_one_chunk(ids, a.M * a.k, a.E, hist, sort);   // (the counters take the place of counts and logits)
  }
}

// ---- small routers: all that stands in front of the experts' GEMMs but the sort ----------------------------------
//
// RMSNorm, activation quantiser, router matmul and selection are four launches' worth of dependent work on few bytes: with a
// router of up to 64 experts over a hidden size of up to 1024 a workgroup can read all of the router's weights itself (66 KB for
// 33 columns of 1024, from L2), so each does the whole chain for its tokens: one launch, no partial sums in memory.
//   Its eight waves take a row's pieces of eight values 64 at a time, square, normalise and quantise them and put them into LDS,
// while the weights travel into registers; then wave w multiplies K block w of all rows (128 values, a quantisation group) with
// up to five fragments of 16 columns (65 in all), the blocks' products meet in LDS, and a wave selects a token's experts.  Sums, blocks and
// instructions are those of rmsnorm_quant_kernel, router_gemm_kernel (where its K slices are 128 long) and route_kernel in their
// order: the same bits.
//   What bounds it: the launch's start and four trips through memory and LDS.  Against the launches that it replaces (us): mini
// layer (33 columns of 1024), 1 token 5.5 / 7.5, 64 7.3 / 9.5, 4096 12.1 / 14.0; behind its norm 1 token 6.0 / 7.9, 200 7.5 /
// 13.1, 1000 8.6 / 14.4; tiny (8 of 512), 100 tokens 4.0 / 7.8.  Sixteen tokens a workgroup at any size: 11.1 for 64 tokens, 13.6
// for 200 behind the norm.  The limits on columns and hidden size are what a wave has registers and a workgroup waves for.
constexpr int kFrontTokens = 16, kFrontWaves = 8, kFrontExperts = 64, kFrontColumns = kFrontExperts + 1, kFrontD = 128 * kFrontWaves;
constexpr int front_lds(int tokens, int D, int N, int E) { return tokens * D * 2 + (tokens * N * (D / 128 + 1) + E) * 4; }
constexpr int kFrontLds = front_lds(kFrontTokens, kFrontD, kFrontColumns, kFrontExperts);   // 70464
struct FrontJob {
  const void* x;
  int x_f32, D, tokens;         // tokens of a workgroup: a power of two up to kFrontTokens
  const float* norm;            // NORM
  float eps;
  const bf16_t *w, *w_extra;    // (E, D) and the shared expert's gate (1, D) or null
  uint8_t* xq;                  // null: no quantisation
  float *sx, *sx_blocked;
  int32_t* chunk_hist;          // [workgroups][E] or null
};

template <int KIND, bool NORM>
__global__ __launch_bounds__(64 * kFrontWaves) void front_kernel(const RouteArgs a, const FrontJob f) {
  extern __shared__ __attribute__((aligned(16))) int lds[];   // [rows' pieces][the K blocks' products][logits][E counts]
  constexpr int GROUPS = (kFrontColumns + 15) / 16, UNITS = kFrontTokens * (kFrontD / 512) / kFrontWaves;
  __shared__ float wave_sum[kFrontTokens][kFrontD / 512];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, fq = lane >> 4;
  const int N = a.src.N, E = a.E, D = f.D, KB = D / 128, P = D / 8, T = f.tokens;
  const int t0 = blockIdx.x * T;
  v4i* pieces = (v4i*)lds;   // piece p of row r at p ^ (r & 7)
  float* products = (float*)(pieces + T * P);
  float* rows = products + KB * T * N;
  int* hist = (int*)(rows + T * N);
  // unit u: pieces [64 (u % per_row), +64) of row u / per_row; wave w has units w, w + 8, ...
  const int per_row = P > 64 ? 2 : 1, units = T * per_row;
  moe_bf16x8 in[UNITS] = {};
  v4f wt[UNITS][2] = {};
#pragma unroll
  for (int i = 0; i < UNITS; ++i) {
    const int u = w + kFrontWaves * i, p = (u & (per_row - 1)) * 64 + lane, t = t0 + (per_row == 2 ? u >> 1 : u);
    if (u < units && p < P && t < a.M) {
      in[i] = load_bf16x8(f.x, f.x_f32, (size_t)t * P + p);
      if (NORM) wt[i][0] = ((const v4f*)f.norm)[2 * p], wt[i][1] = ((const v4f*)f.norm)[2 * p + 1];
    }
  }
  v4i b[GROUPS][4];
  if (w < KB) front_weights(b, f.w, f.w_extra, E, N, D, w);
  if (f.chunk_hist && tid < E) hist[tid] = 0;
  if (NORM) {
#pragma unroll
    for (int i = 0; i < UNITS; ++i) {
      const int u = w + kFrontWaves * i;
      if (u >= units) break;
      const float ss = wave_sum_f32(front_squares(in[i]));
      if (lane == 0) wave_sum[per_row == 2 ? u >> 1 : u][u & (per_row - 1)] = ss;
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < UNITS; ++i) {
    const int u = w + kFrontWaves * i;
    if (u >= units) break;
    const int p = (u & (per_row - 1)) * 64 + lane, r = per_row == 2 ? u >> 1 : u;
    if (NORM) {
      const float total = per_row == 2 ? __fadd_rn(wave_sum[r][0], wave_sum[r][1]) : wave_sum[r][0];
      front_norm(in[i], total, D, f.eps, wt[i]);
    }
    if (p < P) pieces[r * P + (p ^ (r & 7))] = __builtin_bit_cast(v4i, in[i]);
  }
  __syncthreads();
  if (w < KB) {
    v4i av[4];
    const int r = fr & (T - 1);   // (rows beyond the tile's: any)
#pragma unroll
    for (int s = 0; s < 4; ++s) av[s] = pieces[r * P + ((w * 16 + 4 * s + fq) ^ (r & 7))];
#pragma unroll
    for (int g = 0; g < GROUPS; ++g) {
      if (16 * g >= N) break;
      const v4f acc = front_products(av, b[g]);
      const int n = 16 * g + fr;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (4 * fq + j < T && n < N) products[(w * T + 4 * fq + j) * N + n] = acc[j];
    }
  }
  __syncthreads();
  for (int i = tid; i < T * N; i += 64 * kFrontWaves) rows[i] = front_logit(products + i, KB, T * N);
  __syncthreads();
  for (int tt = w; tt < min(T, a.M - t0); tt += kFrontWaves) {
    const float* row = rows + tt * N;
    if (a.src.out_logits && lane < E) a.src.out_logits[(size_t)(t0 + tt) * E + lane] = row[lane];
    if (lane == 0 && a.src.shared_gate && N > E) a.src.shared_gate[t0 + tt] = front_gate(row[E]);
    const int chosen = KIND == ROUTE_SOFTMAX ? route_softmax_token<1>(a, row, t0 + tt).expert : route_grouped_token<1>(a, row, t0 + tt).expert;
    if (f.chunk_hist && lane < a.k) atomicAdd(&hist[chosen], 1);
  }
  if (f.xq) {   // (nobody in this launch waits for the codes)
#pragma unroll
    for (int i = 0; i < UNITS; ++i) {
      const int u = w + kFrontWaves * i;
      if (u >= units) break;
      const int p = (u & (per_row - 1)) * 64 + lane, t = t0 + (per_row == 2 ? u >> 1 : u);
      float scale_inv;
      const uint2 out = front_codes(in[i], scale_inv);
      if (p < P && t < a.M) {
        ((uint2*)f.xq)[(size_t)t * P + p] = out;
        if ((p & 15) == 0) {
          f.sx[(size_t)t * KB + p / 16] = scale_inv;
          if (f.sx_blocked) f.sx_blocked[(size_t)(p / 16) * a.M + t] = scale_inv;
        }
      }
    }
  }
  if (f.chunk_hist) {
    __syncthreads();
    if (tid < E) f.chunk_hist[(size_t)blockIdx.x * E + tid] = hist[tid];
  }
}

constexpr int kCUs = 256;

}  // namespace

int moe_route_check(int routing, const RouteArgs& a) {
  const LogitSource& src = a.src;
  const int M = a.M, E = a.E, k = a.k;
  MOE_REQUIRE(M == 0 || ((src.logits || src.partial) && a.idx && a.w), MOE_ERR_NULL, "route: null pointer");
  MOE_REQUIRE(!src.partial || (src.splits >= 1 && src.N >= E), MOE_ERR_BAD_SHAPE, "route: bad partial-sum layout");
  MOE_REQUIRE(M >= 0 && E >= 1 && E <= 1024, MOE_ERR_BAD_SHAPE, "route: need 1 <= E <= 1024, got E=%d M=%d", E, M);
  MOE_REQUIRE(k >= 1 && k <= 32 && k <= E, MOE_ERR_BAD_SHAPE, "route: need 1 <= k <= min(32,E), got k=%d E=%d", k, E);
  if (routing == MOE_ROUTING_SIGMOID_GROUPED) {
    MOE_REQUIRE(a.n_group >= 1 && a.n_group <= 64 && E % a.n_group == 0, MOE_ERR_BAD_SHAPE,
                "route: n_group=%d must divide E=%d and be <= 64", a.n_group, E);
    MOE_REQUIRE(a.topk_group >= 1 && a.topk_group <= a.n_group, MOE_ERR_BAD_SHAPE,
                "route: topk_group=%d out of range for n_group=%d", a.topk_group, a.n_group);
    MOE_REQUIRE(k <= a.topk_group * (E / a.n_group), MOE_ERR_BAD_SHAPE,
                "route: k=%d exceeds the %d experts of the kept groups", k, a.topk_group * (E / a.n_group));
  }
  return MOE_OK;
}

namespace {

template <int KIND, bool SORT_HERE>
void launch_route(int vpl, dim3 grid, dim3 block, size_t lds, hipStream_t s, const RouteArgs& a, const RouteJob& job,
                  const QuantJob& q, const PermuteOut& o) {
  if (vpl <= 1) hipLaunchKernelGGL((route_kernel<1, KIND, SORT_HERE>), grid, block, lds, s, a, job, q, o);
  else if (vpl <= 2) hipLaunchKernelGGL((route_kernel<2, KIND, SORT_HERE>), grid, block, lds, s, a, job, q, o);
  else if (vpl <= 4) hipLaunchKernelGGL((route_kernel<4, KIND, SORT_HERE>), grid, block, lds, s, a, job, q, o);
  else if (vpl <= 8) hipLaunchKernelGGL((route_kernel<8, KIND, SORT_HERE>), grid, block, lds, s, a, job, q, o);
  else hipLaunchKernelGGL((route_kernel<16, KIND, SORT_HERE>), grid, block, lds, s, a, job, q, o);
}

}  // namespace

int moe_route_impl(int routing, const RouteArgs& a, const QuantJob* quant, const PermuteOut* sort, void* permute_ws,
                   size_t permute_ws_bytes, moe_stream_t stream) {
  if (int rc = moe_route_check(routing, a)) return rc;
  MOE_REQUIRE((!quant && !sort) || a.M > 0, MOE_ERR_BAD_SHAPE, "route: nothing to carry a quantisation or a sort with");
  MOE_REQUIRE(!sort || (permute_ws && permute_ws_bytes >= moe_permute_workspace_bytes(a.M, a.k, a.E)), MOE_ERR_WORKSPACE_TOO_SMALL,
              "route: permutation workspace too small");
  MOE_REQUIRE(!sort || (long long)a.M * a.k < (1ll << 31), MOE_ERR_BAD_SHAPE, "route: M*k overflows int32");
  if (a.M == 0) return MOE_OK;
  const int R = a.M * a.k;
  RouteJob job{};
  // One workgroup takes a batch whose partial sums (if any) it can add about as fast as many would: the sort needs no
  // launch of its own then.
  const bool sort_here = sort && route_sorts_here(a.M, a.k, a.src.partial) && R <= kSmallRows &&
                  (!a.src.partial || (long long)a.M * a.src.N * a.src.splits <= 65536);
  const bool one_chunk = R <= kSmallRows;   // the placing kernel counts such a list itself
  // Tokens per workgroup: one per wave, or one in all while there are few and their partial sums are the work (router
  // of 4096 x 256 and routing, one token against four: 64 tokens 11.8 / 15.0 us, 1024 21.4 / 22.5, 2048 24.7 / 22.4).
  int tpb = a.src.partial && a.M <= 1024 ? 1 : 4;
  bool counts = sort && !sort_here && !one_chunk;
  if (counts) {
    // A workgroup that counts its selections for the sort owns a histogram, and those are few (moe_permute_max_chunks):
    // 256, a workgroup of 16 waves on every CU, up to 256 experts, 64 for 1024.  Where that leaves CUs idle, the
    // selections are counted by the sort's own first launch.  Ready logits, counted here / there: 300 experts, 1024
    // tokens 39.4 / 36.3 us of a small layer, 8192 87.2 / 84.7; 512 experts, 4096 tokens 59.3 / 53.2; 1024 experts, 512
    // tokens 53.9 / 52.4, 8192 163.7 / 93.3 (partial sums 231 / 114).  256 experts, 8192 tokens: 82.6 / 81.7.
    const int max_chunks = moe_permute_max_chunks(a.E);
    if (max_chunks < kCUs && a.M > 4 * max_chunks) counts = false;
    else if ((a.M + max_chunks - 1) / max_chunks > tpb) tpb = (a.M + max_chunks - 1) / max_chunks;
  }
  if (sort_here) tpb = a.M;
  // Eight tokens a workgroup and more take sixteen waves, or eight where the launch carries the quantiser: a workgroup of
  // sixteen fits beside another on a CU only when all of its slots are free, and the quantiser's blocks stood waiting.
  // Qwen3-MoE, 4096 tokens 14.7 -> 11.0 us, 4000 of the mini layer 9.4 -> 8.4, 8000 of the tiny layer 10.0 -> 9.3 (four waves
  // 16.1, 11.9 and 13.9); without it 2500 tokens of the mini layer from f32 take 66.7 us with sixteen, 68.4 with eight.
  //   A token whose partial sums are the work and that has a CU to itself: a thread a column (513 columns in 32 slices: the
  // launch 10.5 -> 9.3 us for 1 token, 12.0 -> 10.6 for 200).
  const bool own_cu = a.src.partial && tpb == 1 && a.M <= kCUs;
  const int threads = sort_here || (tpb >= 8 && !quant) || (own_cu && a.src.N > 512) ? 1024 : tpb >= 8 || (own_cu && a.src.N > 256) ? 512 : 256;
  job.tokens_per_block = tpb;
  job.blocks = (a.M + tpb - 1) / tpb;
  job.chunk_hist = counts ? (int32_t*)permute_ws : nullptr;
  job.batch = tpb;
  size_t ints = (sort_here ? kSmallRows : 0) + (size_t)a.E;
  size_t tail = 0;
  if (a.src.partial) {
    const int room = 12288 / a.src.N;   // 48 KB of logits (N <= 1025)
    const int waves = threads / MOE_WAVE;
    job.batch = waves < room ? waves : room;
    if (job.batch > tpb) job.batch = tpb;
    tail = (size_t)job.batch * a.src.N;
  }
  if (sort_here && moe_place_lds_ints(a.E) > tail) tail = moe_place_lds_ints(a.E);
  const size_t lds = (ints + tail) * sizeof(int);
  const QuantJob q = quant ? *quant : QuantJob{};
  const PermuteOut o = sort ? *sort : PermuteOut{};
  const dim3 grid(job.blocks + (quant ? moe_quant_blocks(q, threads) : 0)), block(threads);
  const int vpl = (a.E + 63) / 64;
  hipStream_t s = (hipStream_t)stream;
  const auto launch = routing == MOE_ROUTING_SOFTMAX ? (sort_here ? launch_route<ROUTE_SOFTMAX, true> : launch_route<ROUTE_SOFTMAX, false>)
                                                      : (sort_here ? launch_route<ROUTE_GROUPED, true> : launch_route<ROUTE_GROUPED, false>);
  launch(vpl, grid, block, lds, s, a, job, q, o);
  if (int rc = moe_check_hip(hipGetLastError(), "route launch")) return rc;
  if (!sort || sort_here) return MOE_OK;
  if (one_chunk) return moe_permute_place(a.idx, R, a.E, kSmallRows, 1, nullptr, o, nullptr, stream);
  if (!counts) return moe_permute_impl(a.idx, a.M, a.k, a.E, o, permute_ws, permute_ws_bytes, nullptr, stream);
  return moe_permute_place(a.idx, R, a.E, tpb * a.k, job.blocks, job.chunk_hist, o, nullptr, stream);
}

// Routers that front_kernel takes: where the K slices of the router's matmul are its K blocks (the same sums), and one workgroup a CU
// has all tokens (4096).  With more of them there are more workgroups than histograms, and the sort counts in a launch of its own.
// Layers of 64 experts, launch by launch / this way (us; 4096 tokens of 1024 behind the norm: 65.8 / 60.5):
//   behind the norm, 4600 of 1024 69.1 / 76.5, 5000 of 640 67.4 / 72.6, 8192 of 512 66.5 / 64.1, 12000 of 256 67.1 / 66.4, 20000 of
// 128 84.0 / 86.1, 65536 of it 189 / 218;
//   without it, 4600 of 1024 60.4 / 62.7, 5000 of 640 58.8 / 59.7, 8192 of 512 58.5 / 57.6, 32000 of 256 101.0 / 96.5; from f32,
// which else needs its rounding stored, 5000 of 640 69.7 / 66.8, 4097 of 1024 72.2 / 66.4;
//   the routing alone, 4600 of 1024 15.1 / 13.1, 32000 of 256 28.5 / 24.1, 65536 of 128 42.1 / 39.8, 262144 132 / 157.
bool moe_front_takes(int M, int D, int E, int N, bool norm, bool x_f32, bool sorted) {
  if (M < 1 || E > kFrontExperts || D < 128 || D > kFrontD || D % 128 || moe_router_k_slice(M, N, D) != 128) return false;
  return M <= kFrontTokens * kCUs || (M <= 32768 && !norm && (!sorted || x_f32 || D <= 512));
}
int moe_front_check(int routing, RouteArgs& a, const FrontArgs& f, bool sorted) {
  const int N = a.E + (f.w_shared_gate ? 1 : 0);
  MOE_REQUIRE(f.x && f.w_router && (!f.w_shared_gate || a.src.shared_gate) && (!f.xq || f.sx), MOE_ERR_NULL, "router: null pointer");
  MOE_REQUIRE(MOE_ALIGNED16(f.x) && MOE_ALIGNED16(f.w_router) && MOE_ALIGNED16(f.w_shared_gate) && MOE_ALIGNED16(f.norm) && MOE_ALIGNED16(f.xq),
              MOE_ERR_BAD_ALIGN, "router: pointers must be 16-byte aligned");
  MOE_REQUIRE(moe_front_takes(a.M, f.D, a.E, N, f.norm, f.x_f32, sorted), MOE_ERR_BAD_SHAPE, "router: not a call for this launch (M=%d D=%d N=%d)", a.M, f.D, N);
  a.src.logits = nullptr, a.src.partial = (const float*)f.w_router, a.src.splits = 1, a.src.N = N;   // (no logits are given, and none are in memory)
  return moe_route_check(routing, a);
}
int moe_front_impl(int routing, RouteArgs a, const FrontArgs& f, const PermuteOut* sort, void* permute_ws, size_t permute_ws_bytes,
                   moe_stream_t stream) {
  if (int rc = moe_front_check(routing, a, f, sort)) return rc;
  const int N = a.src.N;
  MOE_REQUIRE(!sort || (permute_ws && permute_ws_bytes >= moe_permute_workspace_bytes(a.M, a.k, a.E)), MOE_ERR_WORKSPACE_TOO_SMALL,
              "route: permutation workspace too small");
  MOE_REQUIRE((long long)a.M * a.k < (1ll << 31), MOE_ERR_BAD_SHAPE, "route: M*k overflows int32");
  MOE_REQUIRE((long long)a.M * f.D * 2 < (1ll << 32), MOE_ERR_BAD_SHAPE, "router: the activations must stay within 4 GB");   // (as moe_router_partials)
  // Tokens of a workgroup: one, or as many as it takes to have one workgroup a CU.
  int tokens = 1;
  while (tokens < kFrontTokens && tokens * kCUs < a.M) tokens *= 2;
  const int R = a.M * a.k, blocks = (a.M + tokens - 1) / tokens;
  const bool one_chunk = R <= kSmallRows, counts = sort && !one_chunk && blocks <= moe_permute_max_chunks(a.E);
  const FrontJob job{f.x, f.x_f32, f.D, tokens, f.norm, f.eps, (const bf16_t*)f.w_router, (const bf16_t*)f.w_shared_gate, f.xq, f.sx, f.sx_blocked,
                     counts ? (int32_t*)permute_ws : nullptr};
  const int lds = front_lds(tokens, f.D, N, a.E);
  auto* kernel = routing == MOE_ROUTING_SOFTMAX ? (f.norm ? front_kernel<ROUTE_SOFTMAX, true> : front_kernel<ROUTE_SOFTMAX, false>)
                                                : (f.norm ? front_kernel<ROUTE_GROUPED, true> : front_kernel<ROUTE_GROUPED, false>);
  static std::atomic<unsigned long long> lds_raised[4] = {};
  if (int rc = moe_raise_lds_limit((const void*)kernel, kFrontLds, lds_raised[(routing == MOE_ROUTING_SOFTMAX ? 0 : 2) + (f.norm ? 1 : 0)])) return rc;
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(64 * kFrontWaves), lds, (hipStream_t)stream, a, job);
  if (int rc = moe_check_hip(hipGetLastError(), "route launch")) return rc;
  if (!sort) return MOE_OK;
  if (one_chunk) return moe_permute_place(a.idx, R, a.E, kSmallRows, 1, nullptr, *sort, nullptr, stream);
  if (!counts) return moe_permute_impl(a.idx, a.M, a.k, a.E, *sort, permute_ws, permute_ws_bytes, nullptr, stream);
  return moe_permute_place(a.idx, R, a.E, tokens * a.k, blocks, (const int32_t*)permute_ws, *sort, nullptr, stream);
}

extern "C" int moe_route_softmax_topk(const float* logits, int M, int E, int k, int renorm,
                                      int32_t* idx, float* w, moe_stream_t stream) {
  const RouteArgs a{LogitSource{logits, nullptr, 0, E, nullptr, nullptr}, nullptr, M, E, k, renorm, 1, 1, 1.f, idx, w};
  return moe_route_impl(MOE_ROUTING_SOFTMAX, a, nullptr, nullptr, nullptr, 0, stream);
}

extern "C" int moe_route_sigmoid_grouped(const float* logits, const float* bias, int M, int E,
                                         int n_group, int topk_group, int k, int renorm,
                                         float routed_scale, int32_t* idx, float* w,
                                         moe_stream_t stream) {
  const RouteArgs a{LogitSource{logits, nullptr, 0, E, nullptr, nullptr}, bias, M, E, k, renorm, n_group, topk_group,
                    routed_scale, idx, w};
  return moe_route_impl(MOE_ROUTING_SIGMOID_GROUPED, a, nullptr, nullptr, nullptr, 0, stream);
}

extern "C" int moe_routing(const void* x_bf16, int M, int D, const void* w_router_bf16, int E, int k, int renorm, int32_t* idx,
                           float* w, void* ws, size_t ws_bytes, moe_stream_t stream) {
  int splits = 0, n_cols = 0;
  if (moe_front_takes(M, D, E, E, false, false, false)) {
    MOE_REQUIRE(ws, MOE_ERR_NULL, "router: null pointer");
    MOE_REQUIRE(MOE_ALIGNED16(ws), MOE_ERR_BAD_ALIGN, "router: pointers must be 16-byte aligned");
    MOE_REQUIRE(ws_bytes >= moe_router_workspace_bytes(M, D, E), MOE_ERR_WORKSPACE_TOO_SMALL, "router: workspace %zu < %zu", ws_bytes,
                moe_router_workspace_bytes(M, D, E));
    const RouteArgs a{LogitSource{}, nullptr, M, E, k, renorm, 1, 1, 1.f, idx, w};
    return moe_front_impl(MOE_ROUTING_SOFTMAX, a, FrontArgs{x_bf16, 0, D, nullptr, 0.f, w_router_bf16, nullptr, nullptr, nullptr, nullptr}, nullptr,
                          nullptr, 0, stream);
  }
  if (int rc = moe_router_partials(x_bf16, M, D, w_router_bf16, E, nullptr, ws, ws_bytes, &splits, &n_cols, stream)) return rc;
  const RouteArgs a{LogitSource{nullptr, (const float*)ws, splits, n_cols, nullptr, nullptr}, nullptr, M, E, k, renorm, 1, 1, 1.f, idx, w};
  return moe_route_impl(MOE_ROUTING_SOFTMAX, a, nullptr, nullptr, nullptr, 0, stream);
}
