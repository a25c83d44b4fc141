// The stable counting sort's placing step as device functions of one workgroup, shared by its own kernel
// (moe_permute.hip) and by the routing kernel of a small batch (moe_route.hip), which sorts what it has just selected.
#pragma once
#include "moe_common.h"

constexpr int kMaxE = 1024;
constexpr int kPlaceThreads = 1024;
constexpr int kPlaceWaves = kPlaceThreads / MOE_WAVE;

// waves that count and place: one counter per expert each, at most 32 KB of LDS in all
__host__ __device__ inline int moe_place_waves(int E) { return E > 512 ? kPlaceWaves / 2 : kPlaceWaves; }
__host__ __device__ inline size_t moe_place_lds_ints(int E) { return (size_t)moe_place_waves(E) * E; }
// ... of a chunk of n entries: as many as have 64 entries to take (every wave's counters are cleared, added up and walked)
__host__ __device__ inline int moe_place_waves(int E, int n) {
  const int most = moe_place_waves(E), filled = (n + MOE_WAVE - 1) / MOE_WAVE;
  return filled < 1 ? 1 : filled < most ? filled : most;
}

#ifdef __HIPCC__
// lanes of this wave whose expert id equals mine (ids < 2^bits); inactive lanes pass id = -1
__device__ __forceinline__ unsigned long long match_any(int id, int bits) {
  unsigned long long m = __ballot(id >= 0);
  for (int b = 0; b < bits; ++b) {
    unsigned long long set = __ballot((id >> b) & 1);
    m &= ((id >> b) & 1) ? set : ~set;
  }
  return id >= 0 ? m : 0ull;
}

__device__ __forceinline__ int ilog2_ceil(int n) { return n <= 1 ? 0 : 32 - __clz(n - 1); }

// Counts or places the entries [first, first + n) of the flat list, wave w a contiguous share of them in flat order, so
// that a wave's own counters and the popcount of the match mask below a lane give stable ranks.  `next` is [waves][E]:
// PLACE false: += the wave's entries per expert; true: next free output position, advanced as entries are placed.
template <bool PLACE>
__device__ __forceinline__ void place_pass(const int32_t* ids, int first, int n, int E, int* next, const PermuteOut& o) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, waves = moe_place_waves(E, n);
  if (wv >= waves) return;
  const int bits = ilog2_ceil(E);
  const int span = (n + waves * MOE_WAVE - 1) / (waves * MOE_WAVE) * MOE_WAVE;   // uniform
  int* mine = next + wv * E;
  for (int i0 = wv * span; i0 < min(n, (wv + 1) * span); i0 += MOE_WAVE) {
    const int i = i0 + lane;
    int id = i < n ? ids[i] : -1;
    if (id >= E) id = -1;   // out-of-range ids are dropped rather than corrupting LDS
    const unsigned long long m = match_any(id, bits);
    const int rank = __popcll(m & ((1ull << lane) - 1ull));
    int pos = -1;   // (a dropped entry has no row)
    if (id >= 0) {
      if (PLACE) pos = mine[id] + rank;             // every lane of a class reads before its leader bumps the counter
      if (rank == 0) mine[id] += __popcll(m);       // (one writer per counter and instruction)
      if (PLACE) {
        const int f = first + i;
        if (o.sort_order) o.sort_order[pos] = f;
        if (o.sorted_token_ids) o.sorted_token_ids[pos] = (int)((unsigned)f / (unsigned)o.k);   // (half the code of a signed division)
      }
    }
    if (PLACE && i < n && o.inv_perm) o.inv_perm[first + i] = pos;
  }
}

// Behind the kept entries, where dropped ones leave the sorted lists without any: zeros, so that whoever walks a list to its
// end stays inside the rows.  (Whole workgroup; kept: entries that have a place.)
__device__ __forceinline__ void zero_list_ends(int kept, int R, const PermuteOut& o) {
  for (int i = kept + (int)threadIdx.x; i < R; i += kPlaceThreads) {
    if (o.sort_order) o.sort_order[i] = 0;
    if (o.sorted_token_ids) o.sorted_token_ids[i] = 0;
  }
}

// The sort of at most kFewRows entries by one workgroup of kPlaceThreads, without counters or barriers: every wave that has
// experts holds all entries, one a lane, and its threads go through them, eight at a time, for their experts' rows and what
// stands in front of them.  An expert that has rows has one tile.  With the counters below the same step of the routing launch
// takes 2.3 to 2.6 us, this way 1.2 for 8 entries and 2.0 for 32 (64: 3.2).
constexpr int kFewRows = 32;   // (no tile is shorter)
__device__ __forceinline__ void permute_few(const int32_t* ids, int n, int E, const PermuteOut& o) {
  const int e = threadIdx.x, lane = e & 63;
  if (e >= ((E + 63) & ~63)) return;   // (whole waves: no expert is theirs)
  int id = lane < n ? ids[lane] : -1;
  if (id >= E) id = -1;   // out-of-range ids are dropped
  const unsigned long long same = match_any(id, ilog2_ceil(E));
  const int rank = __popcll(same & ((1ull << lane) - 1ull)), first = id >= 0 && rank == 0;
  int rows = 0, start = 0, tile = 0, pos = rank;   // (pos: of this lane's entry)
  for (int j0 = 0; j0 < n; j0 += 8) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {   // (lanes past the last entry hold -1, as dropped ones: above every expert)
      const unsigned other = (unsigned)__builtin_amdgcn_readlane(id, j0 + i);
      const int new_expert = __builtin_amdgcn_readlane(first, j0 + i);
      const bool before = other < (unsigned)e;
      rows += other == (unsigned)e;
      start += before;
      tile += before ? new_expert : 0;
      pos += other < (unsigned)id;
    }
  }
  if (e < E) {
    o.group_sizes[e] = rows;
    o.group_offsets[e] = start;
    if (e == E - 1) o.group_offsets[E] = start + rows;
    if (o.tl.tiles && rows && tile < o.tl.max_tiles) o.tl.tiles[tile] = TileEntry{e | 1 << 10, start, rows, tile};
  }
  if (o.tl.tiles) {
    const int all = min((int)__popcll(__ballot(first)), o.tl.max_tiles);
    if (e == 0) moe_tile_even_shares(o.tl.hdr, all, all);
  }
  if (e < n && id >= 0) {
    if (o.sort_order) o.sort_order[pos] = e;
    if (o.sorted_token_ids) o.sorted_token_ids[pos] = (int)(((float)e + 0.5f) * __builtin_amdgcn_rcpf((float)o.k));   // e / k
  }
  if (e < n && o.inv_perm) o.inv_perm[e] = id >= 0 ? pos : -1;   // (a dropped entry has no row)
  zero_list_ends((int)__popcll(__ballot(id >= 0)), n, o);   // (n <= 32: threads of the first wave)
}

// The whole sort of one chunk (n entries starting at flat index 0) in one workgroup of kPlaceThreads; ids may be in
// LDS.  next: moe_place_lds_ints(E) ints of LDS.  The caller synchronises before the call (ids written, LDS free).
__device__ __forceinline__ void permute_one_chunk(const int32_t* ids, int n, int E, int* next, const PermuteOut& o) {
  if (n <= kFewRows) return permute_few(ids, n, E, o);
  const int e = threadIdx.x, waves = moe_place_waves(E, n);
  for (int i = threadIdx.x; i < waves * E; i += kPlaceThreads) next[i] = 0;
  __syncthreads();
  place_pass<false>(ids, 0, n, E, next, o);
  __syncthreads();
  int rows = 0;
  if (e < E)
#pragma unroll 4
    for (int w = 0; w < waves; ++w) rows += next[w * E + e];
  const int nt = o.tl.tiles ? moe_tile_count(rows, o.tl.tile_rows) : 0;
  int row_start = rows, tile_start = nt, rows_all, tiles_all;
  moe_scan_1024(row_start, tile_start, rows_all, tiles_all);
  if (e < E) {
    int run = row_start;
#pragma unroll 4
    for (int w = 0; w < waves; ++w) {
      const int c = next[w * E + e];
      next[w * E + e] = run;
      run += c;
    }
    o.group_sizes[e] = rows;
    o.group_offsets[e] = row_start;
    if (e == E - 1) o.group_offsets[E] = row_start + rows;
    if (o.tl.tiles) {
      for (int t = 0; t < nt; ++t)
        if (tile_start + t < o.tl.max_tiles) o.tl.tiles[tile_start + t] = TileEntry{e | nt << 10, row_start, rows, tile_start};
      if (e == 0) {
        const int all = min(tiles_all, o.tl.max_tiles);
        moe_tile_even_shares(o.tl.hdr, all, all);
      }
    }
  }
  zero_list_ends(rows_all, n, o);
  __syncthreads();
  place_pass<true>(ids, 0, n, E, next, o);
}
#endif
