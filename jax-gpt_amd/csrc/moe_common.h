// Shared device/host helpers for the gfx950 MoE kernels.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <stdint.h>

#include "moe_hip.h"

#define MOE_WAVE 64
#define MOE_QBLOCK 128  // scale granularity along K (and N for weights)
#define MOE_FP8_MAX 448.0f

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned short bf16_t;  // raw bf16 bits

// host side: record an error message for moe_last_error() and return the code
int moe_set_error(int code, const char* fmt, ...);
int moe_check_hip(hipError_t e, const char* what);

// hipFuncSetAttribute applies to the current device: remember, per kernel, on which devices the dynamic LDS limit
// has been raised (bit d of the mask = device d; safe to call from several host threads).
inline int moe_raise_lds_limit(const void* kernel, int bytes, std::atomic<unsigned long long>& done_mask) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return moe_check_hip(e, "hipGetDevice");
  const unsigned long long bit = 1ull << (dev & 63);
  if (done_mask.load(std::memory_order_acquire) & bit) return MOE_OK;
  e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e != hipSuccess) return moe_check_hip(e, "raising the dynamic LDS limit");
  done_mask.fetch_or(bit, std::memory_order_release);
  return MOE_OK;
}

// ---- work list of the grouped GEMMs ----
// One entry per row tile, in [expert][tile] order; every entry carries its EXPERT's row range and the index of the
// expert's first tile, from which a workgroup derives its own tile and column block (moe_gemm.hip).  The list
// depends on the group sizes and the tile height only, so the gate/up and the down GEMM of a layer share it.
struct TileHeader {
  int n_tiles;
  // The first n_static tiles are dealt to the XCDs in fixed shares (xcd_q).  The rest -- the smallest experts, last in
  // the list -- are a pool that the workgroups of every XCD draw from once their share is done, an item at a time
  // through pool_next (one counter per GEMM of the layer: gate/up, down; the list's builder sets them to zero, so a
  // list serves one launch of each).  An XCD that is ahead takes more of the pool: it evens out what the fixed
  // shares cannot know (the XCDs' paces differ by a few per cent, and so does the cost estimate behind the shares).
  int n_static;
  int pool_next[2];
  // Where the work of XCD k begins, as a tile position with 20 fraction bits (xcd_q[0] = 0, xcd_q[8] = n_static << 20);
  // a GEMM with ncb column blocks per row tile gives XCD k the items [xcd_q[k] * ncb >> 20, xcd_q[k + 1] * ncb >> 20).
  long long xcd_q[9];
  long long pad2;
};
constexpr int kTileQBits = 20;
// The pool holds at most TileList::pool_tiles tiles, and an XCD may draw up to twice its eighth of it: the grouped GEMM
// launches this many workgroups per XCD beyond its fixed share for a GEMM of ncb column blocks per row tile.
//   It is max_tiles / 16 (a pool of max_tiles / 8 and up to 4 or 6 tail rounds measured 0.5-1 % slower), or a quarter of
// max_tiles for lists of a few rounds of long items (moe_gemm_pool_tiles) if the groups are uneven: fixed shares cannot end
// together there, and a draw (some 1 us) is little beside an item.  Expert-parallel shard, 32 experts of 7168 x 2048 with
// Zipf(1.2) rows, 1/16, 1/4 and 1/2 of max_tiles: 1600 rows 265 / 253 / 248 us, 2400 294 / 279 / 268, 4800 355 / 337 / 359,
// 6400 451 / 398 / 409, 8000 470 / 449 / 455, 12000 620 / 604 / 605, 16384 766 / 761 / 768.
constexpr int kTailRounds = 3, kWideTailRounds = 8;   // rounds of the ranking (8 experts each) that end a bin or go to the pool
__host__ __device__ inline int moe_pool_workgroups(long long pool_items) { return (int)(pool_items >> 2) + 1; }
// The grouped GEMM launches ceil(max_tiles * ncb / 8) + 2 workgroups per XCD: a split whose largest share stays
// within max_tiles / 8 tiles fits whatever ncb is (max_tiles is a worst case over all group sizes, so a real list
// is usually a good deal shorter and its shares fit with room to spare).
__host__ __device__ inline long long moe_xcd_share_cap_q(int max_tiles) {
  return ((long long)max_tiles << kTileQBits) >> 3;
}
struct TileEntry {
  int expert_tiles;   // expert (10 bits), then its number of row tiles (a list holds at most 2^25 / 288 of them)
  int row_start, rows, first_tile;
};
struct TileList {
  int max_tiles;
  int pool_tiles;     // more than max_tiles / 16: only where the groups are uneven
  int rows;           // of all groups
  int tile_rows;      // rows of a full tile: a multiple of 32, at most kTileRows; or kTallTileRows, see moe_tile_rows_voted
  TileHeader* hdr;
  TileEntry* tiles;
  int ncb[2];         // column blocks per row tile of the GEMMs that will read the list (0: none), ...
  int round_q[2];     // ... and 32 work items in tiles, with kTileQBits fraction bits
};
// An expert with `rows` rows gets ceil(rows / tile_rows) row tiles whose heights, counted in units of 32 rows, differ by
// at most one: no tile computes more than 31 rows of padding, and tiles that share a weight slab take about the same
// time per K step and walk it together, so the later reader finds it in L2.
constexpr int kTileRows = 288, kTallTileRows = 320;   // (the latter: moe_tile_rows_voted)
__host__ __device__ inline int moe_tile_count(int rows, int tile_rows) { return rows <= 0 ? 0 : (int)((unsigned)(rows + tile_rows - 1) / (unsigned)tile_rows); }
// A list that may have tall tiles has them where these give every expert with rows the same number, n = ceil(R / E / 320), and
// full tiles would give some expert one more: a few tiles beyond whole rounds are a round of their own.  (Uneven groups gain
// nothing by the height, and their longest items end last: Qwen3-MoE with normal offsets of 2 on the logits, 2500 to 8192 tokens,
// +2 to +7 % with tall tiles throughout.)  The list's builder adds its experts' votes up: the first from the low half, the second
// from the high one.
__host__ __device__ inline int moe_tall_tiles(int R, int E) { return (int)((unsigned)(R / E + kTallTileRows - 1) / (unsigned)kTallTileRows); }
__host__ __device__ inline int moe_tall_vote(int rows, int n) {
  return rows <= 0 ? 0 : moe_tile_count(rows, kTallTileRows) != n ? 1 : moe_tile_count(rows, kTileRows) > n ? 1 << 16 : 0;
}
__host__ __device__ inline int moe_tile_rows_voted(int tile_rows, int votes) {
  return tile_rows <= kTileRows ? tile_rows : (votes & 0xffff) == 0 && votes ? kTallTileRows : kTileRows;
}
// first row (relative to the expert's first) and row count of tile t of nt
__host__ __device__ inline void moe_tile_span(int rows, int nt, int t, int& start, int& count) {
  if (nt == 1) {   // (integer division costs some forty instructions on this hardware: the one-tile case takes none)
    start = 0;
    count = rows;
    return;
  }
  const int units = (rows + 31) >> 5;
  const int base = units / nt, extra = units - base * nt;
  start = (t * base + (t < extra ? t : extra)) << 5;
  const int full = (base + (t < extra ? 1 : 0)) << 5;
  count = full < rows - start ? full : rows - start;
}
#ifdef __HIPCC__
// Where an expert's tiles go in the work list.  The grouped GEMM deals contiguous eighths of the list to the 8 XCDs
// (tiles that share a weight slab then share an L2), so the eighths should cost about the same: with group sizes
// as skewed as a biased router makes them, natural expert order leaves one XCD with up to a tenth more work than the
// average, and the launch ends with its slowest XCD.  The experts are therefore ranked by size (in units of 32 rows)
// and dealt to eight bins in snake order (0..7, 7..0, ...); the list holds bin after bin.
// Called by every thread of a workgroup of 1024, or of a single wave (WAVE: up to 64 experts); thread e owns expert e (rows = nt = 0
// where there is none); lds_a and lds_b are an int a thread in LDS.  Returns the index of expert e's first tile and writes the list header.
//
// The header's XCD shares are cut by cost, not by count: a row tile of u 32-row units costs about 8 + u (measured:
// 63 us for a 32-row tile of the gate/up GEMM against 112 us for a 256-row one, and the same ratio for the down
// GEMM), and equal counts left the XCD with the tallest tiles some 3 % more work than the average.  All tiles of an
// expert cost alike, so a cut inside an expert sits at the same fraction of its items as of its cost.
//
// One workgroup, between two launches that wait for it, so it is written for few steps: the ranking is a counting sort
// over size classes, an expert's place in the list follows from its rank in closed form, and the tiles and cost in
// front of it are one scan over the list.  (Comparing every expert with every other took 10, 17 and 45 us at 128, 256
// and 512 experts; this takes 4.)
__device__ inline int moe_tile_cost(int rows, int tiles) { return 8 * tiles + ((rows + 31) >> 5); }   // (< 2^31 for 2^32 / 128 rows)
__device__ inline void moe_tile_even_shares(TileHeader* hdr, int n_static, int n_tiles) {   // one thread
  hdr->n_tiles = n_tiles;
  hdr->n_static = n_static;
  hdr->pool_next[0] = hdr->pool_next[1] = 0;
  for (int k = 0; k <= 8; ++k) hdr->xcd_q[k] = (((long long)n_static << kTileQBits) * k) >> 3;
}
// Inclusive sum over a wave's lanes by DPP: shifts inside the rows of 16, then the rows' totals broadcast to the rows
// behind.  (A shuffle is a trip through LDS, some 100 cycles and twice the code a step, and a chain of three scans
// stands in front of the grouped GEMMs.  With it and with the counters of filled waves alone in the placing step the
// placing launch takes 3.8 us for 512 entries over 8 experts, 4.6 before; 10.2 for 32768 over 128, 11.6 before; the
// routing launch that sorts one token of 32 experts 6.2, 7.4 before.)
template <int CTRL, int ROWS> __device__ __forceinline__ int moe_dpp_add(int v) {
  return v + __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xF, false);   // (0 from outside the row)
}
__device__ __forceinline__ int moe_row_scan(int v) {
  v = moe_dpp_add<0x111, 0xF>(v);   // row_shr:1, 2, 4, 8
  v = moe_dpp_add<0x112, 0xF>(v);
  v = moe_dpp_add<0x114, 0xF>(v);
  return moe_dpp_add<0x118, 0xF>(v);
}
__device__ __forceinline__ int moe_wave_scan(int v) {
  v = moe_row_scan(v);
  v = moe_dpp_add<0x142, 0xA>(v);   // row_bcast:15 into rows 1 and 3
  return moe_dpp_add<0x143, 0xC>(v);   // row_bcast:31 into rows 2 and 3
}
// exclusive sums of (a, b) over the workgroup's 1024 threads, and the totals
__device__ __forceinline__ void moe_scan_1024(int& a, int& b, int& all_a, int& all_b) {
  __shared__ int wave_a[16], wave_b[16];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int in_a = moe_wave_scan(a), in_b = moe_wave_scan(b);
  if (lane == 63) wave_a[wv] = in_a, wave_b[wv] = in_b;
  __syncthreads();
  const int sum_a = moe_row_scan(wave_a[lane & 15]), sum_b = moe_row_scan(wave_b[lane & 15]);   // every row the same
  all_a = __builtin_amdgcn_readlane(sum_a, 15);
  all_b = __builtin_amdgcn_readlane(sum_b, 15);
  a = in_a - a + (wv ? __builtin_amdgcn_readlane(sum_a, (wv - 1) & 15) : 0);
  b = in_b - b + (wv ? __builtin_amdgcn_readlane(sum_b, (wv - 1) & 15) : 0);
  __syncthreads();   // (the wave totals may be overwritten)
}
// the same over the workgroup's threads: 1024, or (WAVE) one wave's
template <bool WAVE> __device__ __forceinline__ void moe_scan_threads(int& a, int& b, int& all_a, int& all_b) {
  if constexpr (!WAVE) return moe_scan_1024(a, b, all_a, all_b);
  const int in_a = moe_wave_scan(a), in_b = moe_wave_scan(b);
  all_a = __builtin_amdgcn_readlane(in_a, 63);
  all_b = __builtin_amdgcn_readlane(in_b, 63);
  a = in_a - a;
  b = in_b - b;
}
template <bool WAVE = false>
__device__ inline int moe_tile_first(int e, int rows, int nt, int* lds_a, int* lds_b, const TileList& l) {
  constexpr int THREADS = WAVE ? MOE_WAVE : 1024;
  TileHeader* const hdr = l.hdr;
  const int max_tiles = l.max_tiles;
  __shared__ long long cut_q[9];
  __shared__ int tail_tiles[kWideTailRounds];   // tiles of the last, last but one, ... round of the ranking
  // rank: largest class first, inside a class in any order (1023 units = the largest class and everything above it)
  const int units = min((rows + 31) >> 5, 1023);
  int rank, nz, all_tiles;   // nz: experts with rows
  if (e < kWideTailRounds) tail_tiles[e] = 0;
  if constexpr (WAVE) {   // bit by bit, the lanes of larger and of equal classes
    unsigned long long larger = 0, equal = __ballot(rows > 0);
    nz = (int)__popcll(equal);
    for (int b = 9; b >= 0; --b) {
      const bool mine = units >> b & 1;
      const unsigned long long set = __ballot(mine);
      if (!mine) larger |= equal & set;
      equal &= mine ? set : ~set;
    }
    rank = (int)(__popcll(larger) + __popcll(equal & ((1ull << e) - 1)));
    all_tiles = __builtin_amdgcn_readlane(moe_wave_scan(nt), 63);
    __syncthreads();
  } else {
    const int cls = rows > 0 ? 1023 - units : 0;
    lds_a[e] = 0;
    __syncthreads();
    const int order = rows > 0 ? atomicAdd(&lds_a[cls], 1) : 0;
    __syncthreads();
    int before = lds_a[e], tiles_to = nt;
    moe_scan_1024(before, tiles_to, nz, all_tiles);
    lds_b[e] = before;
    __syncthreads();
    rank = lds_b[cls] + order;
  }
  const int nr = (nz + 7) >> 3;   // rounds that hold a non-empty expert
  int tail = nr / 4 < kTailRounds ? nr / 4 : kTailRounds;   // (3 rounds = 24 experts over the 8 bins; 6 measured no better)
  int pool_most = max_tiles >> 4;
  const long long all_items = (long long)all_tiles * (l.ncb[0] ? l.ncb[0] : l.ncb[1]);
  const bool whole = all_items == 256 || all_items == 512;   // one or two full rounds: equal shares end together, draws do not
  if (l.pool_tiles > pool_most && !whole && (WAVE ? __any((long long)rows * nz > 2ll * l.rows) : __syncthreads_or((long long)rows * nz > 2ll * l.rows))) {   // (an expert of twice the mean)
    tail = nr > kWideTailRounds ? kWideTailRounds : nr - 1;
    pool_most = l.pool_tiles;
  }
  const int round = rank >> 3;
  if (rows > 0 && round >= nr - tail) atomicAdd(&tail_tiles[nr - 1 - round], nt);
  __syncthreads();
  // The pool: as many of the tail rounds, from the last one, as fit the launch's spare workgroups.
  int pooled = 0;
  for (int t = 0, sum = 0; t < tail; ++t) {
    sum += tail_tiles[t];
    if (sum > pool_most) break;
    pooled = t + 1;
  }
  const int n_fixed = pooled ? (nr - pooled) * 8 : nz;   // experts in fixed shares; the others, last in rank, are the pool
  int at = rank;                                         // place in the list
  if (rank < n_fixed) {
    // Inside a bin the experts alternate between the large and the small end of the ranking (largest, smallest,
    // second largest, ...): tall tiles are matrix work on lines that mostly hit L2, short tiles are weight streams
    // from HBM, and a launch that runs them side by side from start to end keeps both busy and its power draw even
    // (largest first throughout: 1.4 % slower on the heavy-tailed DeepSeek-V3 routing, 4 % on the Qwen3-MoE case).
    // The smallest experts of a bin stay at its end (those that the pool does not take): the launch ends with its
    // shortest items.
    const int mixed = nr - tail;
    auto position = [&](int r) { return r >= mixed ? r : r < (mixed + 1) / 2 ? 2 * r : 2 * (mixed - 1 - r) + 1; };
    const int bin = (round & 1) ? 7 - (rank & 7) : rank & 7;
    // full rounds give every bin one expert; a last round of `part` experts gives one to some bins
    const int full = n_fixed >> 3, part = n_fixed & 7;
    const bool odd = full & 1;
    const bool has_part = odd ? bin >= 8 - part : bin < part;
    at = bin * full + (odd ? max(0, bin - (8 - part)) : min(bin, part)) + position(round) -
         (part && !has_part && position(full) < position(round) ? 1 : 0);
  }
  lds_a[e] = 0;   // (the class counts were read before the scan's barriers, lds_b's prefixes before the last one)
  lds_b[e] = 0;
  __syncthreads();
  if (rows > 0) {
    lds_a[at] = nt;
    lds_b[at] = at < n_fixed ? moe_tile_cost(rows, nt) : 0;   // (the pool has no part in the shares)
  }
  __syncthreads();
  int tiles_before = lds_a[e], cost_before = lds_b[e], total, cost_all;
  moe_scan_threads<WAVE>(tiles_before, cost_before, total, cost_all);
  lds_a[e] = tiles_before;
  lds_b[e] = cost_before;
  __syncthreads();
  const int first = lds_a[at & (THREADS - 1)], mine_before = lds_b[at & (THREADS - 1)];
  const int fixed_tiles = n_fixed < THREADS ? lds_a[n_fixed] : total;
  // cut k sits where the cost of the fixed shares reaches k/8 of their whole: inside exactly one expert, whose
  // thread places it
  if (rows > 0 && at < n_fixed) {
    const long long mine = (long long)moe_tile_cost(rows, nt) * 8;
    for (int k = 1; k < 8; ++k) {
      const long long d = (long long)cost_all * k - (long long)mine_before * 8;   // (cost units x 8)
      if (d >= 0 && d < mine)   // (float: the cut need not be exact, only inside this expert's tiles)
        cut_q[k] = ((long long)first << kTileQBits) + (long long)((float)d / (float)mine * (float)nt * (float)(1 << kTileQBits));
    }
  }
  __syncthreads();
  if (e == 0) {
    const int n = total < max_tiles ? total : max_tiles;
    const int ns = fixed_tiles < n ? fixed_tiles : n;
    cut_q[0] = 0;
    cut_q[8] = (long long)ns << kTileQBits;
    bool fits = ns > 0 && total <= max_tiles;
    // A launch of one or two rounds over the CUs ends with whole items: an XCD with 33 of them takes as long as one with
    // 64.  There no share may hold more than that many rounds' items.  (8 experts of 1024 rows of the tiny layer, 256 items:
    // 67.5 -> 59.3 us; 9 tiles x 28 columns of 768 to 192 rows 46.8 -> 36.7.  Three rounds of unequal tiles lose by it, an
    // expert-parallel shard of 8000 rows 481 -> 490.)
    long long cap = moe_xcd_share_cap_q(max_tiles);
    for (int g = 0; g < 2; ++g) {
      const long long rounds = ((long long)n * l.ncb[g] + 255) >> 8;
      if (rounds == 1 || rounds == 2) cap = min(cap, rounds * l.round_q[g]);
    }
    for (int k = 0; k < 8 && fits; ++k) fits = cut_q[k + 1] - cut_q[k] <= cap;
    moe_tile_even_shares(hdr, ns, n);   // (a share beyond what the launch provides workgroups for: equal counts always fit)
    if (fits)
      for (int k = 0; k <= 8; ++k) hdr->xcd_q[k] = cut_q[k];
  }
  return first;
}
#endif

// Where the routing kernels take a token's logits from: an (M, E) array, or the router matmul's split-K partial
// sums [splits][M][N] (N = E, + 1 when the shared expert's gate is the last column), which they add in slice order
// and round to bf16 themselves -- the logits then never travel through memory unless out_logits asks for them.
struct LogitSource {
  const float* logits;    // (M, E), used when partial is null
  const float* partial;   // [splits][M][N] or null
  int splits, N;
  float* out_logits;      // optional (M, E) copy of what the kernel ranked (partial mode only)
  float* shared_gate;     // (M) sigmoid of column E, written in partial mode when N > E
};
int moe_router_partials(const void* x_bf16, int M, int D, const void* w_router_bf16, int E,
                        const void* w_shared_gate_bf16, void* ws, size_t ws_bytes, int* splits_used, int* n_cols,
                        moe_stream_t stream);
int moe_router_k_slice(int M, int N, int D);   // K elements of a slice
// RMSNorm, activation quantiser (row-major scales) and router matmul in one launch, for the calls that it takes (N as above)
bool moe_norm_router_takes(int M, int D, int N, int x_f32);
int moe_norm_router_partials(const void* x, int x_f32, const float* weight, float eps, int M, int D, const void* w_router_bf16,
                             int E, const void* w_shared_gate_bf16, uint8_t* xq, float* sx, void* ws, size_t ws_bytes,
                             int* splits_used, int* n_cols, moe_stream_t stream);
// An activation quantisation (moe_quant_device.h): blocks of blockDim.x 16-byte pieces, in a launch of its own or
// behind the routing kernel's own blocks.
struct QuantJob {
  const void* x;        // (R, K) bf16, or f32 (x_f32), which is rounded to bf16 first
  int x_f32;
  void* x_bf16;         // optional (R, K) copy of the rounded f32 values
  long long n_pieces;   // R * K / 8
  int groups_per_row;   // K / 128
  int R;
  uint8_t* xq;
  float* sx;
  float* sx_blocked;    // optional (K/128, R) copy of the scales
};
inline unsigned moe_quant_blocks(const QuantJob& q, int threads) { return (unsigned)((q.n_pieces + threads - 1) / threads); }
int moe_quant_act_job(const void* x, int x_f32, void* x_bf16, int R, int K, uint8_t* xq, float* sx, float* sx_blocked, QuantJob* job);
// Batches up to this many (token, slot) entries are one chunk, and their few, short row tiles are listed in plain
// expert order with equal XCD shares.
constexpr int kSmallRows = 2048;
// What the placing launch of a list of several chunks writes besides (a pointer to both, as these arguments' size is read cold by every
// routing and placing launch)
struct ScaleGather {   // the activation scales of the sorted rows, block-major
  const float* sx;     // (tokens, KB)
  int KB;
  float* out;          // (KB, R)
};
struct PlaceMore {
  const TileList* tl_down;     // a list of its own for the down GEMM, or null: it reads PermuteOut::tl
  const ScaleGather* gather;   // or null
};
// How the routed gate/up GEMM finds its activation scales: block-major in sorted order (gathered; placed: by the placing launch) or in the
// quantiser's rows.  forked: the quantiser may run beside the sort
struct ScalePlan { bool gathered, placed; };
ScalePlan moe_scale_plan(int R, int E, int D, int I, bool forked);
// What the sort by expert writes (sort_order, sorted_token_ids, inv_perm: null to skip; tl.tiles null: no work list).
struct PermuteOut {
  int32_t *group_sizes, *group_offsets, *sorted_token_ids, *sort_order, *inv_perm;
  int k;
  TileList tl;
  const PlaceMore* more;   // or null; batches of more than kSmallRows entries only; read by the host
};
// One routing call: the selection, and with it (optional) an activation quantisation and the sort by expert.
struct RouteArgs {
  LogitSource src;
  const float* bias;   // sigmoid_grouped only, or null
  int M, E, k, renorm;
  int n_group, topk_group;
  float routed_scale;
  int32_t* idx;
  float* w;
};
int moe_route_check(int routing, const RouteArgs& a);   // what the routing launches refuse
int moe_route_impl(int routing, const RouteArgs& a, const QuantJob* quant, const PermuteOut* sort, void* permute_ws,
                   size_t permute_ws_bytes, moe_stream_t stream);
// The same behind the router's matmul, the quantiser and, with norm, the RMSNorm, all in its one launch (small routers; N: columns
// with the shared expert's gate).  a.src: out_logits and shared_gate alone.
struct FrontArgs {
  const void* x;    // (M, D) bf16, or f32 (x_f32), which is rounded to bf16 first
  int x_f32, D;
  const float* norm;
  float eps;
  const void *w_router, *w_shared_gate;
  uint8_t* xq;      // optional: codes, scales and the scales' (D / 128, M) copy
  float *sx, *sx_blocked;
};
bool moe_front_takes(int M, int D, int E, int N, bool norm, bool x_f32, bool sorted);   // sorted: a sort of the selections follows
int moe_front_check(int routing, RouteArgs& a, const FrontArgs& f, bool sorted);   // what the launch refuses; completes a.src
int moe_front_impl(int routing, RouteArgs a, const FrontArgs& f, const PermuteOut* sort, void* permute_ws, size_t permute_ws_bytes,
                   moe_stream_t stream);
// chunks of the flat list that get a histogram each, at most
int moe_permute_max_chunks(int E);
// the sort's second launch: chunk_hist [n_chunks][E]; or, n_chunks == 1 and chunk_hist null, all of it (quant: carried along)
int moe_permute_place(const int32_t* idx, int R, int E, int chunk, int n_chunks, const int32_t* chunk_hist, const PermuteOut& o,
                      const QuantJob* quant, moe_stream_t stream);
// grouped GEMMs with an optional pre-built tile list in ws (moe_gemm.hip); the extern "C" entry points build their
// own.  moe_gemm_tile_list describes the list the GEMMs of (R rows, E experts) expect in ws, so that the permutation
// kernels, which hold every expert's row range anyway, can write it (moe_permute_impl) and no launch is spent on it.
// tile_rows: moe_gemm_tile_rows of the GEMMs that will read it.
// kb: fewest K steps of these GEMMs.
int moe_gemm_tile_list(int R, int E, int tile_rows, int ncb_gateup, int ncb_down, int kb, void* ws, size_t ws_bytes, TileList* list);
// Rows of a full tile for R rows in E groups and, in the same launches, dense_rows rows of a dense group; [0] gate/up,
// [1] down: column blocks per row tile and K steps (0: that GEMM does not read the list).
struct TileShape {
  int R, E;
  int max_rows;   // that a group may have
  int ncb[2], kb[2];
  int dense_rows, dense_ncb[2];
};
int moe_gemm_tile_rows(const TileShape& t);
// ... of the down GEMM's own list, where gate/up's list has tiles of list_rows, or 0: they share that one
int moe_gemm_down_tile_rows(const TileShape& t, int list_rows);
// the activation quantisers with an optional second copy of the scales, block-major in row order ((K/128, R): what
// GemmScales{1, R} reads) -- spares the shared expert of a large batch the separate transposition
// (x_f32: x holds f32 values, rounded to bf16 first)
int moe_quant_act_impl(const void* x, int x_f32, void* x_bf16, int R, int K, uint8_t* xq, float* sx, float* sx_blocked,
                       moe_stream_t stream);
int moe_rmsnorm_quant_impl(const void* x, int x_f32, const float* weight, float eps, int M, int D, void* normed_bf16,
                           uint8_t* xq, float* sx, float* sx_blocked, moe_stream_t stream);
// the combine with the residual and the output in bf16 or (io_f32) f32, the output rounded to bf16 either way
// (E > 0: inv_perm holds the selections, and y's rows stand where these do: none for a selection outside [0, E))
int moe_combine_impl(const void* y_bf16, const float* w, const int32_t* inv_perm, int E, const void* shared_bf16, const float* shared_gate,
                     const void* residual, int io_f32, int M, int k, int D, void* out, moe_stream_t stream);
// the whole sort; its first launch carries the quantisation, if any
int moe_permute_impl(const int32_t* idx, int M, int k, int E, const PermuteOut& o, void* ws, size_t ws_bytes, const QuantJob* quant,
                     moe_stream_t stream);
// Where the grouped GEMMs find an activation scale and put an h scale, in floats: scale of (row, 128-wide K block kb)
// = s[row * in_row + kb * in_kb].  The public entry points use the row-major arrays of the quantisers ({K/128, 1});
// moe_forward hands large batches block-major arrays in row-list order ({1, R}, in_listed = true: indexed by the
// position in the row list, not through row_ids), because a K step then reads its 256 row scales from 8 lines
// instead of 256 (a 4-byte read costs the vector L1 a whole line request: -2 to -3 % GEMM time).
struct GemmScales {
  int in_row, in_kb;
  bool in_listed;
  int out_row, out_cb;   // gate/up only: scale of (row, column block cb) of h = sh[row * out_row + cb * out_cb]
  bool out_through;      // set by the launch: the output's stores go through the L2 at once
};
inline GemmScales moe_row_major_scales(int K, int I) { return GemmScales{K / 128, 1, false, I / 128, 1}; }
// Operands of one grouped GEMM.  Gate/up: w0 = gate, w1 = up, K = D, N = I, out = h codes, out_scale = h scales; down:
// w0 = down, K = I, N = D, out = y (w1, sw1, out_scale and row_ids null).
struct GemmOperands {
  const uint8_t* xq;
  const float* sx;
  const int32_t* row_ids;
  const uint8_t* w0;
  const float* sw0;
  const uint8_t* w1;
  const float* sw1;
  int K, N;
  void* out;
  float* out_scale;
  GemmScales sc;
};
// the routed experts: R rows in E groups through a work list in ws, which the launch builds unless it is there already (list_tile_rows)
struct RoutedGemm {
  GemmOperands op;
  const int32_t* group_offsets;
  int E, R;
  void* ws;
  size_t ws_bytes;
  int list_tile_rows, list_pool_tiles;   // of the list that is there already, or 0: none is
  const int32_t* ids = nullptr;          // the selections (flat, k a token) where the launch reads them itself: no list,
  int k = 0;                             // no group_offsets; rows of gate/up's activations are tokens, all others flat indices
};
// rows of a full tile of such launches, or 0: the GEMMs read a list
int moe_gemm_scan_rows(const TileShape& t, bool from_memory);
// one group of all rows (the shared expert): no list, no workspace
struct DenseGemm {
  GemmOperands op;
  int rows;
};
// Whether three projections of this many bytes come from memory on every call, or from the memory-side cache (256 MB).
inline bool moe_gemm_from_memory(long long projection) { return 3 * projection > (192ll << 20); }
// The checks of a GEMM launch's operands (gate/up or down), for a route that reads them without that launch.
int moe_gemm_check(const GemmOperands& op, int rows, int E, bool down);
// One launch for either or both (nullptr: none); both: the routed list has to be there.
int moe_gemm_gateup_impl(const RoutedGemm* routed, const DenseGemm* dense, moe_stream_t stream);
int moe_gemm_down_impl(const RoutedGemm* routed, const DenseGemm* dense, moe_stream_t stream);

#define MOE_REQUIRE(cond, code, ...) \
  do {                               \
    if (!(cond)) return moe_set_error(code, __VA_ARGS__); \
  } while (0)
#define MOE_ALIGNED16(p) ((((uintptr_t)(p)) & 15u) == 0)

// ---- device helpers -------------------------------------------------------

__device__ __forceinline__ float bf16_to_f32(bf16_t b) { return __uint_as_float(((unsigned)b) << 16); }

__device__ __forceinline__ bf16_t f32_to_bf16(float f) {  // round-to-nearest-even
  unsigned u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (bf16_t)((u >> 16) | 0x40);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (bf16_t)(u >> 16);
}

// two f32 -> two bf16 (RNE) in one dword, low half first: the hardware's packed conversion
__device__ __forceinline__ unsigned pack2_bf16(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2_hw __attribute__((ext_vector_type(2)));
  const bf16x2_hw b = __builtin_convertvector((f32x2){lo, hi}, bf16x2_hw);
  return __builtin_bit_cast(unsigned, b);
}

struct alignas(16) moe_bf16x8 { bf16_t v[8]; };
// eight neighbouring values as bf16: 16 bytes of bf16, or 32 of f32 rounded (piece p of an array)
__device__ __forceinline__ moe_bf16x8 load_bf16x8(const void* x, int is_f32, size_t p) {
  if (!is_f32) return ((const moe_bf16x8*)x)[p];
  const v4f lo = ((const v4f*)x)[2 * p], hi = ((const v4f*)x)[2 * p + 1];
  moe_bf16x8 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r.v[i] = f32_to_bf16(lo[i]), r.v[4 + i] = f32_to_bf16(hi[i]);
  return r;
}

// scale = 448/amax (1 when the group is all zero); both quotients are IEEE-rounded
__device__ __forceinline__ void fp8_scales(float amax, float& scale, float& scale_inv) {
  scale = amax > 0.f ? __fdiv_rn(MOE_FP8_MAX, amax) : 1.0f;
  scale_inv = __fdiv_rn(1.0f, scale);
}

// four f32 -> four e4m3fn codes (RNE), clamped to +-448 first
__device__ __forceinline__ unsigned pack4_e4m3(float a, float b, float c, float d) {
  a = fminf(fmaxf(a, -MOE_FP8_MAX), MOE_FP8_MAX);
  b = fminf(fmaxf(b, -MOE_FP8_MAX), MOE_FP8_MAX);
  c = fminf(fmaxf(c, -MOE_FP8_MAX), MOE_FP8_MAX);
  d = fminf(fmaxf(d, -MOE_FP8_MAX), MOE_FP8_MAX);
  int v = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
  v = __builtin_amdgcn_cvt_pk_fp8_f32(c, d, v, true);
  return (unsigned)v;
}

// exp and sigmoid as a fixed sequence of individually rounded f32 operations (no fused multiply-add), which a
// CPU can repeat bit for bit; files that use them are compiled with -ffp-contract=off
__device__ __forceinline__ float exp_det(float x) {
#pragma clang fp contract(off)
  x = fminf(fmaxf(x, -87.0f), 88.0f);
  float n = rintf(__fmul_rn(x, 1.44269504088896341f));
  float r = __fsub_rn(x, __fmul_rn(n, 0.693145751953125f));
  r = __fsub_rn(r, __fmul_rn(n, 1.42860682030941723212e-6f));
  float p = 1.9875691500e-4f;
  p = __fadd_rn(__fmul_rn(p, r), 1.3981999507e-3f);
  p = __fadd_rn(__fmul_rn(p, r), 8.3334519073e-3f);
  p = __fadd_rn(__fmul_rn(p, r), 4.1665795894e-2f);
  p = __fadd_rn(__fmul_rn(p, r), 1.6666665459e-1f);
  p = __fadd_rn(__fmul_rn(p, r), 5.0000001201e-1f);
  float r2 = __fmul_rn(r, r);
  float y = __fadd_rn(__fmul_rn(p, r2), r);
  y = __fadd_rn(y, 1.0f);
  float two_n = __uint_as_float((unsigned)((int)n + 127) << 23);
  return __fmul_rn(y, two_n);
}

__device__ __forceinline__ float sigmoid_det(float x) {
  return __fdiv_rn(1.0f, __fadd_rn(1.0f, exp_det(-x)));
}

// ---- global -> LDS copies without registers in between -------------------------------------------------------
// The copies are inline assembly on purpose: when the compiler knows that an instruction writes LDS from
// memory it makes every later LDS read wait for ALL outstanding memory operations, which would empty the
// prefetch queue at every K step.  Completion is tracked by hand instead (wait_vm + barrier); these are the
// only vector-memory operations inside the K loop.  The LDS destination of lane l is m0 + l * size; the
// source address is a uniform 64-bit base (scalar registers) + a per-lane 32-bit byte offset.
__device__ __forceinline__ void dma16(const uint8_t* base, unsigned off, uint8_t* l) {
  const unsigned m0v = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)l);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(m0v), "v"(off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void dma4(const uint8_t* base, unsigned off, uint8_t* l) {
  const unsigned m0v = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)l);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(m0v), "v"(off), "s"(base) : "memory", "m0");
}
// the same two copies with the LDS destination given as a 32-bit LDS address (uniform): keeps 64-bit generic
// pointers to LDS, which the compiler holds in vector register pairs, out of the loops that issue the copies
__device__ __forceinline__ void dma16(const uint8_t* base, unsigned off, unsigned lds_addr) {
  const unsigned m0v = __builtin_amdgcn_readfirstlane(lds_addr);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(m0v), "v"(off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void dma16_nt(const uint8_t* base, unsigned off, unsigned lds_addr) {   // for lines that are read once
  const unsigned m0v = __builtin_amdgcn_readfirstlane(lds_addr);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(m0v), "v"(off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void dma4(const uint8_t* base, unsigned off, unsigned lds_addr) {
  const unsigned m0v = __builtin_amdgcn_readfirstlane(lds_addr);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(m0v), "v"(off), "s"(base) : "memory", "m0");
}
// a 16-byte store; `through`: the L2 passes it on at once instead of when the line falls out of it
__device__ __forceinline__ void store16(v4i* dst, v4i v, bool through) {
  if (through) asm volatile("global_store_dwordx4 %0, %1, off sc1" ::"v"(dst), "v"(v) : "memory");
  else *dst = v;
}
__device__ __forceinline__ void wait_lgkm0() { __builtin_amdgcn_s_waitcnt(0xC07F); }   // lgkmcnt = 0, other counters untouched
template <int N> __device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));   // vmcnt = N, other counters untouched
}
// the same copy with a full 64-bit address per lane (rows that live in different allocations)
__device__ __forceinline__ void dma16_addr(const void* lane_addr, uint8_t* l) {
  const unsigned m0v = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)l);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(m0v), "v"(lane_addr) : "memory", "m0");
}
