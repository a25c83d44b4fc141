// Stable counting sort of the flat (token, slot) list by expert id.
//
// Replaces jax_gpt/models/qwen35/moe.py:58-80 (_sort_and_group: argsort of the
// flat expert ids, the scatter-add histogram, and the gathers of token ids).
// Two launches, all integer work (one launch when the list fits one chunk):
//   1. per-chunk histograms (inside moe_forward the routing kernel has counted its own selections already);
//   2. every chunk's workgroup adds up the chunk histograms itself -- all of them for the experts' row ranges, those
//      in front of it for its own first positions -- and places its entries: earlier waves' counts through LDS,
//      earlier lanes by popcount of the match mask.  One more workgroup writes the group sizes and offsets and the
//      grouped GEMMs' work list at the same time.
// A launch of this size is bound by its start, not by its work (an idle launch takes 3 us, each chain of dependent
// cold loads 1-2 us more), so the chunk count is capped to keep the second launch's redundant reads of the histograms
// (chunks x E counts per workgroup, at most 256 KB from L2) cheaper than a third launch that would scan them once.
#include <type_traits>

#include "moe_common.h"
#include "moe_permute_device.h"
#include "moe_quant_device.h"

namespace {

constexpr int kHistThreads = 256;

__global__ __launch_bounds__(kHistThreads) void hist_kernel(const int32_t* __restrict__ ids, int R, int E, int chunk,
                                                           int n_chunks, int32_t* __restrict__ chunk_hist, const QuantJob quant) {
  if ((int)blockIdx.x >= n_chunks) {   // the blocks behind quantise the activations (QuantJob)
    moe_quant_act_block(quant, (int)blockIdx.x - n_chunks);
    return;
  }
  extern __shared__ int hist[];  // E
  for (int e = threadIdx.x; e < E; e += kHistThreads) hist[e] = 0;
  __syncthreads();
  const int first = blockIdx.x * chunk, n = min(chunk, R - first);
  for (int i = threadIdx.x; i < n; i += kHistThreads) {
    const int id = ids[first + i];
    if (id >= 0 && id < E) atomicAdd(&hist[id], 1);  // out-of-range ids are dropped rather than corrupting LDS
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += kHistThreads) chunk_hist[(size_t)blockIdx.x * E + e] = hist[e];
}

// TWO: there is a second work list, l2, for the same experts (a kernel of its own: with the choice between them in all launches Qwen3-MoE of
// 4096 tokens took 1.2 us more).  GATHER: the entries' activation scales are written to their places too, and what that needs stands where
// the quantiser's arguments do, which a list of several chunks has none of (as an argument more, Qwen3-MoE of 1000 tokens +0.6 us).
template <bool TWO, bool GATHER>
__global__ __launch_bounds__(kPlaceThreads) void place_kernel(const int32_t* __restrict__ ids, int R, int E, int chunk,
                                                             int n_chunks, const int32_t* __restrict__ chunk_hist,
                                                             const PermuteOut o, const std::conditional_t<GATHER, ScaleGather, QuantJob> job,
                                                             const TileList l2) {
  extern __shared__ int smem[];   // [waves][E]
  if constexpr (!TWO && !GATHER)
    if (n_chunks == 1) {
      if (blockIdx.x > 0) {   // the blocks behind quantise the activations (QuantJob)
        moe_quant_act_block(job, (int)blockIdx.x - 1);
        return;
      }
      permute_one_chunk(ids, R, E, smem, o);
      return;
    }
  __shared__ int total[kMaxE], before[kMaxE];
  const int e = threadIdx.x;
  // chunk; workgroup 0 (started first) does the experts' side, and one behind it the second list
  const int c = (int)blockIdx.x - (TWO ? 2 : 1);
  const bool second = TWO && blockIdx.x == 1;
  const TileList l = second ? l2 : o.tl;
  total[e] = 0;
  before[e] = 0;
  const int first = c * chunk, n = c < 0 ? 0 : min(chunk, R - first);
  const int waves = moe_place_waves(E, n);
  for (int i = e; i < waves * E; i += kPlaceThreads) smem[i] = 0;
  __syncthreads();
  // thread (part, e2) adds expert e2's counts in chunks part, part + parts, ...: independent coalesced loads
  int epad = MOE_WAVE;
  while (epad < E) epad <<= 1;
  const int parts = kPlaceThreads / epad, e2 = e & (epad - 1), part = e / epad;
  if (e2 < E) {
    int all = 0, mine = 0;
#pragma unroll 8
    for (int k = part; k < n_chunks; k += parts) {
      const int v = chunk_hist[(size_t)k * E + e2];
      all += v;
      mine += k < c ? v : 0;
    }
    if (all) atomicAdd(&total[e2], all);
    if (mine) atomicAdd(&before[e2], mine);
  }
  if (c >= 0) place_pass<false>(ids + first, first, n, E, smem, o);
  __syncthreads();
  const int rows = total[e];
  int row_start = rows, vote = o.tl.tile_rows > kTileRows ? moe_tall_vote(rows, moe_tall_tiles(R, E)) : 0, rows_all, votes;
  moe_scan_1024(row_start, vote, rows_all, votes);
  if (c < 0) {
    if (!second && e < E) {
      o.group_sizes[e] = rows;
      o.group_offsets[e] = row_start;
      if (e == E - 1) o.group_offsets[E] = row_start + rows;
    }
    if (!second) zero_list_ends(rows_all, R, o);
    if (l.tiles) {   // the grouped GEMMs' row tiles, an expert's tiles side by side (uniform branch)
      const int nt = moe_tile_count(rows, moe_tile_rows_voted(l.tile_rows, votes));
      const int at = moe_tile_first(e, rows, nt, total, before, l);
      for (int t = 0; t < nt; ++t)
        if (at + t < l.max_tiles) l.tiles[at + t] = TileEntry{e | nt << 10, row_start, rows, at};
    }
    return;
  }
  if (e < E) {
    int run = row_start + before[e];
#pragma unroll 4
    for (int w = 0; w < waves; ++w) {
      const int v = smem[w * E + e];
      smem[w * E + e] = run;
      run += v;
    }
  }
  __syncthreads();
  place_pass<true>(ids + first, first, n, E, smem, o);
  if constexpr (GATHER) {   // sixteen lanes an entry; its place from where the pass above has put it
    __syncthreads();
    for (int i = first + (e >> 4); i < first + n; i += kPlaceThreads / 16) {
      const int pos = o.inv_perm[i];
      const float* row = job.sx + (size_t)((unsigned)i / (unsigned)o.k) * job.KB;
      if (pos >= 0)
        for (int kb = e & 15; kb < job.KB; kb += 16) job.out[(size_t)kb * R + pos] = row[kb];
    }
  }
}

}  // namespace

int moe_permute_max_chunks(int E) {
  const int c = 65536 / E;
  return c < 64 ? 64 : c > 256 ? 256 : c;
}

extern "C" size_t moe_permute_workspace_bytes(int M, int k, int E) {
  (void)M, (void)k;
  return E > 0 ? (size_t)moe_permute_max_chunks(E) * E * sizeof(int32_t) + 256 : 256;
}

// Gathering the activation scales is a launch (5 us); reading them row-major costs the gate/up GEMM a line per row and K
// step, which short tiles of a short launch hide.  Gathered against not: Qwen3-MoE (K blocks x column blocks = 96), 300
// tokens 124.6 / 121.9 us, 1024 145.5 / 142.9, 1500 163.0 / 162.4, 2000 189.0 / 191.3; mini layer, 1100 tokens 52.9 / 51.8;
// DeepSeek-V3 (896), 300 tokens 1176 / 1179, 1100 1530 / 1547.
//   Few scales are written by the placing launch (the quantiser is in front of it where nothing is forked): no launch, but writes of
// four bytes.  Launch by launch / this way: tiny, 1100 tokens 36.2 / 33.9, 8192 76.7 / 75.2; mini sublayer, 2000 52.0 / 50.8, 9000 133.1 / 131.8;
// Qwen3-MoE, 1600 165.4 / 162.4, 2000 (256 K scales) 179.8 / 176.4, 4096 243.6 / 245.8; rows of 32 scales, full layer, 600 1016 / 1019, 1000
// 1046 / 1050; of 56, DeepSeek-V3, 300 and 777 even.
ScalePlan moe_scale_plan(int R, int E, int D, int I, bool forked) {
  const long long scales = (long long)R * (D / 128);
  const bool gathered = R > kSmallRows && (R > 96ll * E || scales * (I / 128) > (1ll << 20));
  return {gathered, gathered && !forked && D <= 2048 && scales <= (1ll << 18)};
}

int moe_permute_place(const int32_t* idx, int R, int E, int chunk, int n_chunks, const int32_t* chunk_hist, const PermuteOut& o,
                      const QuantJob* quant, moe_stream_t stream) {
  MOE_REQUIRE(n_chunks > 1 || !o.more, MOE_ERR_BAD_SHAPE, "permute: a list of one chunk has no second work list and gathers no scales");
  const PlaceMore more = o.more ? *o.more : PlaceMore{};
  const bool places = R > 0 && (o.sorted_token_ids || o.sort_order || o.inv_perm);
  const unsigned blocks = n_chunks > 1 ? (places ? n_chunks : 0) + (more.tl_down ? 2 : 1) : 1 + (quant ? moe_quant_blocks(*quant, kPlaceThreads) : 0);
  const dim3 grid(blocks), block(kPlaceThreads);
  const size_t lds = moe_place_lds_ints(E) * sizeof(int);
  hipStream_t s = (hipStream_t)stream;
  const TileList l2 = more.tl_down ? *more.tl_down : TileList{};
  if (more.gather)
    hipLaunchKernelGGL((more.tl_down ? place_kernel<true, true> : place_kernel<false, true>), grid, block, lds, s, idx, R, E, chunk, n_chunks, chunk_hist, o,
                       *more.gather, l2);
  else
    hipLaunchKernelGGL((more.tl_down ? place_kernel<true, false> : place_kernel<false, false>), grid, block, lds, s, idx, R, E, chunk, n_chunks, chunk_hist, o,
                       quant ? *quant : QuantJob{}, l2);
  return moe_check_hip(hipGetLastError(), "permute launch");
}

extern "C" int moe_permute(const int32_t* idx, int M, int k, int E, int32_t* group_sizes,
                           int32_t* group_offsets, int32_t* sorted_token_ids, int32_t* sort_order,
                           int32_t* inv_perm, void* ws, size_t ws_bytes, moe_stream_t stream) {
  return moe_permute_impl(idx, M, k, E, PermuteOut{group_sizes, group_offsets, sorted_token_ids, sort_order, inv_perm, k,
                                                   TileList{}, nullptr}, ws, ws_bytes, nullptr, stream);
}

int moe_permute_impl(const int32_t* idx, int M, int k, int E, const PermuteOut& o, void* ws, size_t ws_bytes, const QuantJob* quant,
                     moe_stream_t stream) {
  MOE_REQUIRE((idx || M == 0) && o.group_sizes && o.group_offsets && ws, MOE_ERR_NULL, "permute: null pointer");
  MOE_REQUIRE(M >= 0 && k >= 1 && E >= 1 && E <= kMaxE, MOE_ERR_BAD_SHAPE,
              "permute: need k >= 1 and 1 <= E <= %d, got M=%d k=%d E=%d", kMaxE, M, k, E);
  MOE_REQUIRE((long long)M * k < (1ll << 31), MOE_ERR_BAD_SHAPE, "permute: M*k overflows int32");
  MOE_REQUIRE(ws_bytes >= moe_permute_workspace_bytes(M, k, E), MOE_ERR_WORKSPACE_TOO_SMALL,
              "permute: workspace %zu < %zu", ws_bytes, moe_permute_workspace_bytes(M, k, E));
  const int R = M * k;
  if (R <= kSmallRows) return moe_permute_place(idx, R, E, kSmallRows, 1, nullptr, o, quant, stream);
  const int max_chunks = moe_permute_max_chunks(E);
  int chunk = (int)(((long long)R + max_chunks - 1) / max_chunks);
  chunk = chunk < 256 ? 256 : chunk;
  const int n_chunks = (int)(((long long)R + chunk - 1) / chunk);
  hipLaunchKernelGGL(hist_kernel, dim3(n_chunks + (quant ? moe_quant_blocks(*quant, kHistThreads) : 0)), dim3(kHistThreads),
                     E * sizeof(int), (hipStream_t)stream, idx, R, E, chunk, n_chunks, (int32_t*)ws, quant ? *quant : QuantJob{});
  return moe_permute_place(idx, R, E, chunk, n_chunks, (const int32_t*)ws, o, nullptr, stream);
}
