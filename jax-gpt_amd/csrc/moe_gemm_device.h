// What the grouped GEMM kernels share: the constants of a work item, and how a workgroup finds its own.
#pragma once
#include <type_traits>

#include "moe_common.h"

// moe_gemm_stream.hip: the launch, and whether it is one for that kernel
struct StreamLaunch {
  GemmOperands routed;
  TileHeader* hdr;
  const TileEntry* tiles;
  int rows;   // of all routed groups
  GemmOperands dense;
  int dense_rows, dense_tiles, dense_blocks;
  bool from_memory;
  unsigned grid;
  int tile_rows;
};
constexpr int kStreamItems = 384;   // fewest work items, and
constexpr int kStreamRows = 128;    // tallest tiles of such a launch
bool moe_gemm_streams(int mode, int tile_rows, long long items);
int moe_gemm_stream_launch(int mode, const StreamLaunch& l, hipStream_t s);

constexpr int BW = 256;       // weight rows per work item
constexpr int BK = 128;       // K step = scale block
constexpr int MODE_GATEUP = 0;
constexpr int MODE_DOWN = 1;
constexpr int MAX_KB = 256;   // K <= 32768
constexpr int W_TILE_BYTES = BW * BK;   // 32 KB

// Weight stages of that kernel's items of up to 32 rows.  The list's own sizes say which: the host knows only what they can be at most.
//  - Gate/up: one where every item runs at once but some CUs have two of them, two where each CU has one or there are more
//    rounds.  32 experts of 7168 x 2048, gate/up + down + combine, one stage / two: 16 of them with rows (256 items) 130 / 115
//    us, 12 120 / 97, 17 142 / 153, 24 163 / 169; Qwen3-MoE, 9 tokens, 53 experts (318 items) 57.5 / 59.1, 33 49.0 / 45.5, 20
//    42.4 / 37.2; full layer, 7 tokens (some 560) 184 / 169.
//  - Down, in lists that may have taller tiles: two while a tile has ten rows or fewer on average, so that most of the
//    stream is theirs.  The same 32 experts, one stage / two: 160 rows in 24 tiles 187 / 178, 264 in 27 198 / 194, 320 in 28 211 /
//    215, 512 in 30 220 / 225; Qwen3-MoE, 80 tokens in 81 tiles 81.8 / 78.5, in 44 63.9 / 65.7; 200 tokens in 128 113.6 / 114.5.
__host__ __device__ inline int moe_stream_depth(int mode, bool short_only, int tiles, int items, int rows) {
  if (mode == MODE_GATEUP) return items > 256 && items <= 512 ? 1 : 2;
  return short_only || rows <= 10 * tiles ? 2 : 1;
}

// epilogue staging tile: 128-byte rows, chunk c of row r at position c ^ (r & 7)
__device__ __forceinline__ int swz(int row, int chunk) { return row * BK + ((chunk ^ (row & 7)) << 4); }

struct Item { int expert, row_start, row_count, col_block, tiles; };

// Column block and row tile of the `local`-th work item of an expert of nt row tiles and ncb column blocks.
__device__ __forceinline__ void expert_item(int local, int nt, int ncb, int& col_block, int& rt) {
  if (nt < 16) {
    col_block = nt == 1 ? local : local / nt;
    rt = local - col_block * nt;
    return;
  }
  // An expert of many row tiles goes through its column blocks once per group of 8 to 11 row tiles: the 32 CUs
  // of an XCD then work on about 8 row tiles x 4 column blocks at a time (12 distinct operand tiles per K step)
  // instead of 32 row tiles of one column block (33 distinct tiles, every CU pulling the same weight lines at
  // once): 32 row tiles per expert ran 19 % slower than 8.  Below 16 tiles a split does not pay (11 tiles as
  // 6 + 5 measured 1 % slower than unsplit).
  const int ng = nt >> 3;
  const int base = nt / ng, extra = nt - base * ng;   // the first `extra` groups hold base + 1 tiles
  const int big = (base + 1) * ncb * extra;
  int sz, l2, t0;
  if (local < big) {
    sz = base + 1;
    const int g = local / (sz * ncb);
    l2 = local - g * sz * ncb;
    t0 = g * sz;
  } else {
    sz = base;
    const int l = local - big, g = l / (sz * ncb);
    l2 = l - g * sz * ncb;
    t0 = extra * (base + 1) + g * sz;
  }
  col_block = l2 / sz;
  rt = t0 + (l2 - col_block * sz);
}

// The work item of this workgroup, by its index; false: none is left.  (The XCD is blockIdx % 8 for dense and routed items
// alike: dense_blocks is a multiple of 8.)
template <int MODE, bool DENSE>
__device__ __forceinline__ bool work_item(Item& item, uint8_t* lds, int N, bool is_dense, TileHeader* hdr,
                                          const TileEntry* __restrict__ tiles, int dense_rows, int dense_tiles, int dense_blocks) {
  const int xcd = blockIdx.x & 7;
  const int ncb = MODE == MODE_GATEUP ? N / 128 : (N + 255) / 256;
  if (is_dense) {
    // contiguous eighths of the items, so that row tiles that share a weight slab run under one L2
    const int nt = dense_tiles, items = nt * ncb;
    const int per = dense_blocks >> 3;
    const int local = xcd * per + (int)(blockIdx.x >> 3);
    if (local >= items) return false;
    int rt, t0, tn;
    expert_item(local, nt, ncb, item.col_block, rt);
    moe_tile_span(dense_rows, nt, rt, t0, tn);
    item.expert = 0;
    item.tiles = nt;
    item.row_start = t0;
    item.row_count = tn;
  } else {
    // work items = (row tile, column block) pairs in [expert][column block][row tile] order, dealt to the 8 XCDs in
    // contiguous ranges of about equal cost (workgroup ids are issued round-robin over XCDs)
    int item_id = (int)((hdr->xcd_q[xcd] * ncb) >> kTileQBits) + (((int)blockIdx.x - (DENSE ? dense_blocks : 0)) >> 3);
    const int share_end = (int)((hdr->xcd_q[xcd + 1] * ncb) >> kTileQBits);
    if (item_id >= share_end) {
      // behind the XCD's fixed share: the pool of the smallest experts' items, drawn one at a time by whoever gets
      // there (TileHeader); an XCD may draw up to twice its eighth of it
      const int pool_first = hdr->n_static * ncb;
      const int pool_items = (hdr->n_tiles - hdr->n_static) * ncb;
      if (pool_items == 0 || item_id - share_end >= moe_pool_workgroups(pool_items)) return false;   // (uniform: the whole workgroup leaves)
      int* slot = (int*)lds;
      if (threadIdx.x == 0) *slot = atomicAdd(&hdr->pool_next[MODE], 1);   // (the one field of the list a GEMM writes)
      __syncthreads();
      const int drawn = *slot;
      __syncthreads();   // (the work item's first copies overwrite the slot)
      if (drawn >= pool_items) return false;
      item_id = pool_first + drawn;
    }
    const TileEntry te = tiles[item_id / ncb];   // entries [first_tile, first_tile + tiles) all describe this expert
    const int nt = te.expert_tiles >> 10;
    int rt, t0, tn;
    expert_item(item_id - te.first_tile * ncb, nt, ncb, item.col_block, rt);
    moe_tile_span(te.rows, nt, rt, t0, tn);
    item.expert = te.expert_tiles & 1023;
    item.tiles = nt;
    item.row_start = te.row_start + t0;
    item.row_count = tn;
  }
  return true;
}

// The end of a work item.  Weight group wi of the 64 / NW has the weight rows {8 NW wi ..} of both halves (gate/up; fragments
// 0 .. NW / 2 - 1 gate, the others up) or {16 NW wi ..} (down); a lane holds, for weight fragment f and activation fragment j,
// the weight rows (fragment base) + 4 * (lane / 16) + {0..3} of tile row j * ROW_STEP + row0.  All of the workgroup calls it,
// done with the LDS that it stages in: gate/up a f32 maximum per weight group and 128 codes a row, down 256 bf16 a row.
// LISTED: row r of the tile is row listed[r] of the output (in LDS behind what the staging takes).
template <int MODE, int NW, int NF, int BM, int ROW_STEP, int THREADS, bool LISTED = false>
__device__ __forceinline__ void item_epilogue(v4f (&acc)[NW][NF], const Item& item, int row0, int wi, uint8_t* lds, int N,
                                              void* __restrict__ out, float* __restrict__ out_scale, const GemmScales& sc,
                                              const int* listed = nullptr) {
  const int tid = threadIdx.x, fq = (tid & 63) >> 4;
  auto out_row = [&](int r) { return (size_t)(LISTED ? listed[r] : item.row_start + r); };
  if (MODE == MODE_GATEUP) {
    constexpr int NG = NW / 2, GROUPS = 8 / NG;
    float* amax_s = (float*)lds;                            // [GROUPS][BM rows]
    uint8_t* tile = lds + GROUPS * BM * sizeof(float);      // [BM rows][128 B], swizzled
#pragma unroll
    for (int j = 0; j < NF; ++j) {
      float m = 0.f;
#pragma unroll
      for (int f = 0; f < NG; ++f)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float g = acc[f][j][r], u = acc[f + NG][j][r];
          float h = g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)) * u;   // (reciprocal to 1 ulp: far inside the fp8 step)
          acc[f][j][r] = h;
          m = fmaxf(m, fabsf(h));
        }
      m = fmaxf(m, __shfl_xor(m, 16, MOE_WAVE));
      m = fmaxf(m, __shfl_xor(m, 32, MOE_WAVE));
      if (fq == 0) amax_s[wi * BM + j * ROW_STEP + row0] = m;
    }
    __syncthreads();
    const int I = N;
    uint8_t* hq = (uint8_t*)out;
#pragma unroll
    for (int j = 0; j < NF; ++j) {
      const int xr = j * ROW_STEP + row0;
      float m = fmaxf(fmaxf(amax_s[xr], amax_s[BM + xr]), fmaxf(amax_s[2 * BM + xr], amax_s[3 * BM + xr]));
      if (GROUPS == 8)
        m = fmaxf(m, fmaxf(fmaxf(amax_s[4 * BM + xr], amax_s[5 * BM + xr]), fmaxf(amax_s[6 * BM + xr], amax_s[7 * BM + xr])));
      float scale, scale_inv;
      fp8_scales(m, scale, scale_inv);
#pragma unroll
      for (int f = 0; f < NG; ++f) {
        int q = 0;   // (|h| <= amax, so the products stay within a rounding of +-448: one median clamps them)
        q = __builtin_amdgcn_cvt_pk_fp8_f32(__builtin_amdgcn_fmed3f(acc[f][j][0] * scale, -MOE_FP8_MAX, MOE_FP8_MAX),
                                            __builtin_amdgcn_fmed3f(acc[f][j][1] * scale, -MOE_FP8_MAX, MOE_FP8_MAX), q, false);
        q = __builtin_amdgcn_cvt_pk_fp8_f32(__builtin_amdgcn_fmed3f(acc[f][j][2] * scale, -MOE_FP8_MAX, MOE_FP8_MAX),
                                            __builtin_amdgcn_fmed3f(acc[f][j][3] * scale, -MOE_FP8_MAX, MOE_FP8_MAX), q, true);
        const int col = wi * (16 * NG) + f * 16 + fq * 4;  // byte column within the 128-wide slab
        *(unsigned*)(tile + swz(xr, col >> 4) + (col & 15)) = q;
      }
      if (wi == 0 && fq == 0 && xr < item.row_count)
        out_scale[out_row(xr) * sc.out_row + (size_t)item.col_block * sc.out_cb] = scale_inv;
    }
    __syncthreads();
    const int ld_chunk = tid & 7, ld_row = tid >> 3;   // THREADS / 8 rows per pass
#pragma unroll
    for (int i = 0; i < (BM + THREADS / 8 - 1) / (THREADS / 8); ++i) {
      const int r = ld_row + THREADS / 8 * i;
      if (r < item.row_count) {
        v4i v = *(const v4i*)(tile + swz(r, ld_chunk));
        v4i* dst = (v4i*)(hq + out_row(r) * I + item.col_block * 128 + ld_chunk * 16);
        store16(dst, v, sc.out_through);
      }
    }
  } else {
    // bf16 tile [BM rows][256 cols] = 512 B per row, 32 chunks of 16 B, swizzled with (row & 7)
    uint8_t* tile = lds;
#pragma unroll
    for (int j = 0; j < NF; ++j) {
      const int xr = j * ROW_STEP + row0;
#pragma unroll
      for (int f = 0; f < NW; ++f) {
        const int col = wi * (16 * NW) + f * 16 + fq * 4;  // output column within the 256-wide slab
        uint2 v;
        v.x = pack2_bf16(acc[f][j][0], acc[f][j][1]);
        v.y = pack2_bf16(acc[f][j][2], acc[f][j][3]);
        const int chunk = col >> 3;  // 8 bf16 per 16-byte chunk
        *(uint2*)(tile + xr * 512 + ((chunk ^ (xr & 7)) << 4) + (col & 7) * 2) = v;
      }
    }
    __syncthreads();
    bf16_t* y = (bf16_t*)out;
    const bool through = sc.out_through;
    const int wrow0 = item.col_block * 256;
    const int c32 = tid & 31, ld_row = tid >> 5;       // THREADS / 32 rows per pass
    const int ncols = min(256, N - wrow0);
#pragma unroll
    for (int i = 0; i < BM / (THREADS / 32); ++i) {
      const int r = ld_row + THREADS / 32 * i;
      if (r < item.row_count && c32 * 8 < ncols) {
        v4i v = *(const v4i*)(tile + r * 512 + ((c32 ^ (r & 7)) << 4));
        v4i* dst = (v4i*)(y + out_row(r) * N + wrow0 + c32 * 8);
        store16(dst, v, through);
      }
    }
  }
}
