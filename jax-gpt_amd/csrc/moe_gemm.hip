// Grouped fp8 GEMMs over ragged expert row ranges on the CDNA4 fp8 matrix cores.
//
// Replaces the three jax.lax.ragged_dot calls of
// jax_gpt/models/qwen35/moe.py:83-87 (_expert_swiglu):
//   MODE_GATEUP: h = silu(x . Wgate[e]^T) * (x . Wup[e]^T), then 1x128 e4m3 quantisation of h
//   MODE_DOWN:   y = h . Wdown[e]^T, bf16
// for the rows [group_offsets[e], group_offsets[e+1]) of every expert e.
//
// Arithmetic.  Both operands are K-contiguous e4m3 with one f32 scale per 128
// K-elements (activations: per row; weights: per 128 rows), so one
// v_mfma_f32_16x16x128_f8f6f4 consumes exactly one scale block: its 16x16 f32
// result is a partial sum that is multiplied by sx[row,kb]*sw[nblk,kb] and
// added to the f32 accumulator on the vector ALU (the matrix unit has no f32
// scale input).  The weight fragment is the MFMA's row operand and the
// activation fragment its column operand, so a lane holds four weight rows of
// ONE activation row: one activation scale per lane per fragment, not four.
//
// Data movement.  A workgroup (8 waves, two per SIMD, one workgroup per CU) owns a
// work item = (expert, <= 288 activation rows, 256 weight rows) and walks K in
// steps of 128 through a ring of LDS stages.  Tiles are copied global -> LDS by
// global_load_lds (no registers in between) ahead of their use, by one wave of
// each SIMD (wave set 0); the other (set 1) only computes.  In
// MODE_GATEUP the 256 weight rows are 128 gate rows + the 128 up rows of the
// same output columns, so silu(g)*u is lane-local and the 1x128 amax stays
// inside the workgroup.  Waves form a 4 x 2 grid: wave (wi, xj) owns weight rows
// {32wi..32wi+31} of each half (GATEUP) or {64wi..64wi+63} (DOWN) against the
// 16-row activation fragments 2j + xj (alternating between the two wave sets, so
// a short tile still splits evenly).
//
// What bounds a work item.  A K step of a full tile moves 68 KB into LDS (76 copy instructions per CU) and holds
// 2304 matrix-core cycles per SIMD.  Skeletons of the loop on all CUs: 3130 TFLOP/s without the copies, 2737 when every
// weight line is an L2 hit, 2615 when four row tiles share a weight slab from memory, 2181 when each streams its own.
// The activation tile is shared by the item's 16 column blocks and comes from L2, the weight tile comes from L2 when a
// neighbouring row tile of the same expert has just fetched it and from HBM or the memory-side cache otherwise (always,
// for an expert of one row tile).  An expert of few rows is therefore a weight stream at the per-CU HBM rate (31 GB/s of
// both tiles, 41 with non-temporal weight copies) whatever the kernel does with its rows; the kernel's part is to keep that
// stream and the large experts' matrix work going side by side on different CUs, and to waste neither.  The copies'
// cost from an L2-hot source is their issue (address generation, back-pressure from the L1) in the instruction stream of
// the waves that feed the matrix core.
//
// Row tiles are listed on the device (build_tiles_kernel here, or the permutation
// kernels inside moe_forward: no host read-back of group sizes); a workgroup's
// work item is a (row tile, column block) pair derived from its index, in
// [expert][column block][row tile] order, and the items are dealt to the 8 XCDs in
// contiguous ranges, so the row tiles and column blocks that share a weight slab
// or an activation tile run together under one L2.  The items of the smallest
// experts (weight streams, nothing to share) are not dealt out: they sit behind
// the eight ranges as a pool from which the workgroups that follow an XCD's range
// draw one item each through a counter (TileHeader), so an XCD that is ahead
// takes more of them.
//
// Launches of many work items of short row tiles are taken by another kernel, with
// the same items, operands and results: moe_gemm_stream.hip (moe_gemm_tile_rows and
// moe_gemm_streams say which).
#include <stdlib.h>

#include <mutex>
#include <type_traits>

#include "moe_gemm_device.h"

// Tile list of moe_gemm_gateup_swiglu_fp8_static: one copy per GPU, held until the process ends.  In host code this
// name is only a handle for hipGetSymbolAddress; kernels get the address that call returns.
static __device__ __align__(256) unsigned char scratch[MOE_STATIC_SCRATCH_BYTES];

namespace {

constexpr int NWAVES = 8;
constexpr int NT = 64 * NWAVES;
constexpr int ROTC = 2;       // MFMA groups by which wave set 1 trails wave set 0 (measured: 1 to 3 within 2 %)

// ---- work list -----------------------------------------------------------

// One workgroup lists the row tiles of every expert (an expert's tiles side by side; which expert where: see
// moe_tile_first); thread e owns expert e.  Up to 8 rows an expert the tiles cost alike: plain expert order and equal XCD
// shares do, for 2.4 us less a launch (expert-parallel shard of 32 experts, 64 rows 178.3 -> 173.3 us, 256 rows 213 ->
// 208; with 800 unevenly spread rows it would be 239 -> 269).
// WAVE: up to 64 experts, in one wave, with no other waves to start and to wait for at every step (32 experts with 16384 rows 8.3 ->
// 6.2 us a launch, 4.8 for 320 rows; their shard, two lists a pass, 320 rows 212 -> 209.5 us, 800 227.5 -> 224.2, 2400 285.2 ->
// 283.8, 16384 even).  Not where an expert's tiles are written by 64 threads.
__host__ __device__ inline bool many_tiles_each(int E, int max_tiles) { return E <= 16 && max_tiles >= 24 * E; }
template <bool WAVE>
__global__ __launch_bounds__(WAVE ? MOE_WAVE : 1024) void build_tiles_kernel(const int32_t* __restrict__ group_offsets, int E, int R, TileList l) {
  __shared__ int s_rows[WAVE ? MOE_WAVE : 1024];
  __shared__ int s_key[WAVE ? MOE_WAVE : 1024];
  const int e = threadIdx.x;
  int start = 0, rows = 0;
  if (e < E) {
    start = group_offsets[e];
    rows = group_offsets[e + 1] - start;
  }
  const int tiles = moe_tile_count(rows, l.tile_rows);
  int first;
  if (R <= 8 * E) {
    int unused = 0, all, unused_all;
    first = tiles;
    moe_scan_threads<WAVE>(first, unused, all, unused_all);
    if (e == 0) moe_tile_even_shares(l.hdr, min(all, l.max_tiles), min(all, l.max_tiles));
  } else {
    first = moe_tile_first<WAVE>(e, rows, tiles, s_rows, s_key, l);
  }
  // An expert of many tiles is written by 64 threads, not by its own (4096 rows of a 512 x 512 down GEMM in 128 tiles: 18.5
  // -> 11.9 us); below some 24 tiles that costs more than it saves (0.2 us).
  if (!WAVE && many_tiles_each(E, l.max_tiles)) {
    __shared__ TileEntry entry[16];
    if (e < E) entry[e] = TileEntry{e | tiles << 10, start, rows, first};
    __syncthreads();
    const int i = e & 15;
    if (i >= E) return;
    const TileEntry te = entry[i];
    for (int t = e >> 4; t < te.expert_tiles >> 10; t += 64)
      if (te.first_tile + t < l.max_tiles) l.tiles[te.first_tile + t] = te;
    return;
  }
  for (int t = 0; t < tiles; ++t)
    if (first + t < l.max_tiles) l.tiles[first + t] = TileEntry{e | tiles << 10, start, rows, first};   // (cannot overflow for consistent offsets)
}

// ---- the kernel ------------------------------------------------------------------------------------------------
//
// LDS = [ring of weight tiles 256 x 128 B][ring of (activation tile 32 XF x 128 B, its 32 XF activation scales)].
// Tiles are row-major with 128-byte rows; the 16-byte chunk c of row r sits at chunk position
// c ^ ((r >> 1) & 7).  A fragment lane (row fr = lane % 16, quarter fq = lane / 16) feeds the
// MFMA with K bytes [16 fq, +16) and [64 + 16 fq, +16) of its row -- the same choice for both
// operands, so the contraction is unchanged -- which makes every ds_read_b128 of a fragment
// conflict-free (measured ~240 B/clk/CU against ~125 B/clk for 32 contiguous bytes per lane).
// global_load_lds_dwordx4 writes LDS base + lane * 16, i.e. one wave instruction fills 8
// consecutive tile rows; the swizzle is applied by choosing which 16-byte piece of the row
// each lane fetches.  No asynchronous load ever targets a register.

// One launch, row tiles of every height.  A work item's row tile (at most 288 rows, 320 with TALL, near-equal cuts of its
// expert) is served by the smallest of nine (ten: TALL) compiled tile classes that holds it -- 32 XF rows, XF = 1 .. 9 MFMA
// groups per wave and K step -- each a branch-free, fully unrolled K loop of its own with its own LDS ring: the
// short classes have short activation tiles and use the room for more stages (256 rows and more: two stages; 160 to 224
// rows: three weight stages, two activation stages; 64 to 128 rows: three stages, copies two steps ahead; 32 rows:
// four stages, three steps ahead), because an item of a few rows only streams its 256 weight rows and lives on the
// bytes it keeps in flight.  Rows past the end of a tile are multiplied like the others (their copies re-read the tile's last
// row) and never stored.
//
// K step of a wave: XF groups; group j = its four weight fragments against activation fragment j (4 MFMAs, results
// in p[0..3]).  The 16 FMAs that scale group j's results into the accumulators are issued between the MFMAs of
// group j + 1 -- FMA quadruple f just before MFMA f, which overwrites p[f] -- so the matrix core works on the next
// group while the vector ALU finishes the last one, with one set of result registers.  The last group of a step is
// finished behind the next step's barrier, while that step's first fragments travel from LDS.
template <int XF, int MODE = MODE_GATEUP, bool ONCE = true> struct Cls {
  static constexpr int BM = 32 * XF, HALF = BM / 2;
  // Two rings: weight tiles (32 KB each) and activation tiles with their scales.  Where 160 KB allow it the weight
  // ring is one stage deeper than the activation ring (160 to 224 rows: three weight stages, two activation
  // stages): the weight tile is the one that may come from HBM, the activation tile is shared by the item's column
  // blocks and comes from L2.  Measured on the loop's skeleton, weights two steps ahead instead of one: 5-7 % on a
  // weight slab that four workgroups share or that a workgroup streams alone, nothing when every line is an L2 hit.
  static constexpr int X_NST = XF >= 5 ? 2 : XF >= 2 ? 3 : 4;
  static constexpr int W_NST = XF >= 8 ? 2 : XF >= 2 ? 3 : 4;
  // A weight stage is read once per step: every wave loads its four weight fragments into registers when it enters
  // the step, and from then on the stage is free.  With W_EARLY the next tenant's copies are issued right there, in
  // the middle of the step, and not behind the next barrier: the weights of step kb + 2 are then in flight while step
  // kb still computes, as if the ring were a stage deeper, in the same LDS.  The weight rows that wave (wi, 0) copies
  // are read by itself and by wave (wi, 1) alone, so the release is a word in LDS between those two (early_flag)
  // and no barrier.  Only the classes of 256 rows and more of the gate/up GEMM, which have no room for a third stage: -4.5 % where
  // every workgroup streams its own weight slab, -3 % where 8 row tiles share one, -1 % on the mixed tile
  // heights of skewed routing; the down GEMM (16 K steps at the DeepSeek-V3 shape) gained 2 % in the first case and
  // lost 1 % in the second, and the classes with three weight stages cannot gain: their copies complete in issue
  // order behind the activation copies of the step before, which must have landed a step earlier.
  static constexpr bool W_EARLY = XF >= 8 && MODE == MODE_GATEUP;
  static constexpr int EARLY_G = 3;   // the group behind which the weight copies of a W_EARLY step begin (2 and 4: within 1 %)
  static constexpr int X_PRE = X_NST - 1, W_PRE = W_NST - 1 + (W_EARLY ? 1 : 0);   // steps that a copy runs ahead of its use
  // The weight copies' cache policy.  ONCE: the item's expert has one row tile (or two that stay close, see
  // grouped_gemm_kernel) and comes from memory (launch()), so that its weight lines are fetched once and marked
  // non-temporal, which leaves the memory-side cache alone.  A read-only stream reaches 7.1 TB/s that way and 6.3 without
  // (4 GiB, any grid); 64 tokens of the DeepSeek-V3 layer went from 1010 to 864 us, gate/up and down at 6.7 TB/s instead
  // of 5.8.
  static constexpr bool W_ONCE = ONCE;
  static constexpr int X_STAGE_S_OFF = BM * BK;                // the scales behind the tile
  // + 256: every copying wave copies 64 scale slots from its first one on (no lane mask, which would cut the
  // unrolled K step into blocks); the surplus lanes rewrite other waves' slots with the same values or land in this pad
  static constexpr int X_STAGE_BYTES = BM * BK + BM * 4 + 256;
  static constexpr int X_RING_OFF = W_NST * W_TILE_BYTES;
  static constexpr int RING_BYTES = X_RING_OFF + X_NST * X_STAGE_BYTES;
  // Only wave set 0 (waves 0-3) issues copies: a copy instruction can hold its wave at the memory pipeline's door
  // while the L1's queue is full, and with one wave of each SIMD never there the matrix core always has a wave that
  // can feed it (2-3 % over all eight waves copying).  Wave v copies 8 weight row groups (the rows that it reads
  // itself), activation row groups v, v + 4, ... and 64 scale slots.
  static constexpr int X_OPS = XF;                     // activation copies per copying wave and step
  static constexpr int S_OPS = BM > 256 ? 2 : 1;       // scale copies: 64 slots each, four waves
  static constexpr int XS_OPS = X_OPS + S_OPS;
  // Result registers of a wave: the FMAs that scale an MFMA's results stand NP MFMAs behind it.  At 320 rows (160 accumulators)
  // two quadruples are what the register file has left; with four 25 values of the K loop spill, with three 10.
  static constexpr int NP = XF >= 10 ? 2 : 4;
  static constexpr bool S_LATE = XF >= 9;              // read a group's scale with its fragment (registers: 144 are accumulators)
  static constexpr int OPS = 8 + XS_OPS;               // + 8 weight row groups
  // Copies complete in the order of their issue, so within a step those with the earlier deadline go first: with
  // the deeper weight ring the activation copies (and scales), then the weights; with rings of one depth the
  // weights first (they are the ones that may miss).
  static constexpr bool X_FIRST = W_PRE > X_PRE;
  static constexpr bool is_w(int i) { return X_FIRST ? i >= XS_OPS : i < 8; }
  static constexpr int w_index(int i) { return X_FIRST ? i - XS_OPS : i; }
  static constexpr bool is_s(int i) { return X_FIRST ? i >= X_OPS && i < XS_OPS : i >= 8 + X_OPS; }
  static constexpr int s_index(int i) { return X_FIRST ? i - X_OPS : i - 8 - X_OPS; }
  static constexpr int x_index(int i) { return X_FIRST ? i : i - 8; }
  // what may still be in flight when a step starts that found every later copy issued: the activation stages and
  // weight stages of the steps after it
  static constexpr int IN_FLIGHT = (X_PRE - 1) * XS_OPS + (W_PRE - 1) * 8;
  // The same count for a step rem = KB - 1 - kb steps from the item's end: the copies issued behind the last one that
  // the step needs (its activation tile and scales, from X_PRE steps back), where a step that is r steps from the
  // end issued activation copies if r >= X_PRE and weight copies if r >= W_PRE.
  static constexpr int allowed(int rem) {
    int n = 0;
    if (X_FIRST && rem + X_PRE >= W_PRE) n += 8;   // the weight copies behind the needed ones in their own step
    for (int r = rem + X_PRE - 1; r > rem; --r) n += (r >= X_PRE ? XS_OPS : 0) + (r >= W_PRE ? 8 : 0);
    return n;
  }
  static_assert(allowed(W_PRE + X_PRE) == IN_FLIGHT, "the steady state of the rule is the count above");
  // copy operations issued after group g: spread over the first SPREAD groups of the step.  Rings of one depth must
  // have the step's copies out early (they land before the next barrier or hold it up); with the deeper weight ring
  // the weight copies have a step more, and an even spread over the whole step is best (all groups against the
  // first three: gate/up -2 to -4 %, down -1 to -3 % on tiles of 160-224 rows; all at once: +2 %)
  static constexpr int SPREAD = X_FIRST ? XF : XF >= 6 ? XF / 2 : XF >= 3 ? 3 : XF;
  // (W_EARLY: the activation copies and scales behind groups 0 .. EARLY_G - 1, the weight copies behind the rest)
  static constexpr int first(int g) {
    if (W_EARLY)
      return g <= 0 ? 0 : g < EARLY_G ? (XS_OPS * g) / EARLY_G : g >= XF ? OPS : XS_OPS + (8 * (g - EARLY_G)) / (XF - EARLY_G);
    return g <= 0 ? 0 : g >= SPREAD ? OPS : (OPS * g) / SPREAD;
  }
};
constexpr int cmax(int a, int b) { return a > b ? a : b; }
constexpr int CLS_RING = cmax(cmax(cmax(cmax(cmax(Cls<10>::RING_BYTES, Cls<9>::RING_BYTES), Cls<8>::RING_BYTES), Cls<7>::RING_BYTES), cmax(Cls<6>::RING_BYTES, Cls<5>::RING_BYTES)),
                              cmax(cmax(Cls<4>::RING_BYTES, Cls<3>::RING_BYTES), cmax(Cls<2>::RING_BYTES, Cls<1>::RING_BYTES)));
constexpr int CLS_WSCALE_OFF = CLS_RING;                       // [2][MAX_KB] weight block scales of the work item
constexpr int CLS_FLAG_OFF = CLS_WSCALE_OFF + 2 * MAX_KB * 4;  // [4] early_flag: the step whose weight fragments wave (wi, 1) holds, + 1
constexpr int CLS_LDS_BYTES = CLS_FLAG_OFF + 16;              // 160016
constexpr int TALL_LDS_BYTES = 160 * 1024;
static_assert(CLS_LDS_BYTES <= TALL_LDS_BYTES, "LDS");
// The epilogues stage their results where the rings were, all of CLS_RING whatever the class's own rings take: gate/up
// four f32 maxima and 128 codes a row, down 256 bf16 a row -- 144 KB at 288 rows, whose rings are 139 KB; at 320 rows 160 KB,
// the scales' and flags' places included.
template <int XF> constexpr bool epilogue_fits(int bytes) {
  return Cls<XF>::BM * (4 * 4 + BK) <= bytes && Cls<XF>::BM * 256 * 2 <= bytes;
}
static_assert(epilogue_fits<9>(CLS_RING) && epilogue_fits<10>(TALL_LDS_BYTES), "the tallest tile's epilogue stages inside the LDS");

// listed (LDS), row_div: with LISTED, row r of the tile is row listed[r] / row_div of the activations and listed[r] of the output.
template <int MODE, int XF, bool ONCE, bool LISTED = false>
__device__ __forceinline__ void item_body(const Item& item, uint8_t* lds, const uint8_t* __restrict__ xq,
                                          const float* __restrict__ sx, const int32_t* __restrict__ row_ids,
                                          const uint8_t* __restrict__ w0, const float* __restrict__ sw0,
                                          const uint8_t* __restrict__ w1, const float* __restrict__ sw1, int K, int N,
                                          void* __restrict__ out, float* __restrict__ out_scale, const GemmScales sc,
                                          const int* listed = nullptr, int row_div = 1) {
  using C = Cls<XF, MODE, ONCE>;
  constexpr int BM = C::BM, HALF = C::HALF;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wi = wave & 3, xj = wave >> 2;
  const int fr = lane & 15, fq = lane >> 4;
  const int KB = K / BK;
  const int e = item.expert;
  const int wrow0 = MODE == MODE_GATEUP ? item.col_block * 128 : item.col_block * 256;

  // ---- copy sources: copying wave cv (waves 0-3; 4-7 compute the same values and never use them) fills the weight
  // rows that the waves wi = cv read (down: tile rows [64 cv, +64); gate/up: [32 cv, +32) of the gate half and of
  // the up half), activation row groups cv, cv + 4, ... and 64 scale slots
  const int drow = lane >> 3, dchunk = lane & 7;
  const int cv = wave & 3;
  const uint8_t* wmat = w0 + (size_t)e * N * K;   // uniform
  const uint8_t* wmat1 = MODE == MODE_GATEUP ? w1 + (size_t)e * N * K : wmat;
  unsigned woff[2];
  {
    int grow = MODE == MODE_GATEUP ? wrow0 + cv * 32 : wrow0 + cv * 64;
    if (MODE == MODE_DOWN && grow >= N) grow = N - 64;   // (a half-full last column block: re-read valid rows)
    const int piece = dchunk ^ (drow >> 1);
    woff[0] = (unsigned)(grow + drow) * (unsigned)K + piece * 16;
    woff[1] = (unsigned)(grow + drow) * (unsigned)K + (piece ^ 4) * 16;
  }
  unsigned xoff[C::X_OPS];
#pragma unroll
  for (int i = 0; i < C::X_OPS; ++i) {
    const int grp = i * 4 + cv;
    const int r = grp * 8 + drow;                              // row within the activation tile
    const int piece = dchunk ^ ((r >> 1) & 7);
    int g = min(r, item.row_count - 1);
    if constexpr (LISTED) {
      g = (int)((unsigned)listed[g] / (unsigned)row_div);
    } else {
      g += item.row_start;
      if (row_ids) g = row_ids[g];
    }
    xoff[i] = (unsigned)g * (unsigned)K + piece * 16;
  }
  // first of the 64 scale slots that this wave copies (a second copy, all four waves the same, where 256 are not all)
  auto sbase = [&](int i) { return i > 0 ? BM - 64 : BM >= 64 ? min(cv * 64, BM - 64) : 0; };
  unsigned soff[C::S_OPS];
#pragma unroll
  for (int i = 0; i < C::S_OPS; ++i) {
    const int p = min(sbase(i) + lane, BM - 1);   // slots past the tile land in the pad
    const int q = p % HALF;
    const int r = 16 * (2 * (q % XF) + p / HALF) + q / XF;
    int g = min(r, item.row_count - 1);
    if constexpr (LISTED) {
      g = (int)((unsigned)listed[g] / (unsigned)row_div);
    } else {
      g += item.row_start;
      if (row_ids && !sc.in_listed) g = row_ids[g];
    }
    soff[i] = (unsigned)g * (unsigned)sc.in_row * 4u;
  }
  const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)lds);
  // copies of step t's operands: weight row group w of this wave, activation row group x, the scales
  auto copy_w = [&](int t, int w) {
    auto dma = [](const uint8_t* base, unsigned off, unsigned l) {
      if constexpr (C::W_ONCE) dma16_nt(base, off, l);
      else dma16(base, off, l);
    };
    if (MODE == MODE_GATEUP)   // row groups 0-3 of the wave's gate rows, then of its up rows (tile rows 128 ..)
      dma((w < 4 ? wmat : wmat1) + (size_t)t * BK + (size_t)(w & 3) * 8 * K, woff[w & 1],
            lds0 + (unsigned)(t % C::W_NST) * W_TILE_BYTES + ((w < 4 ? 0 : 16) + cv * 4 + (w & 3)) * 1024u);
    else
      dma(wmat + (size_t)t * BK + (size_t)w * 8 * K, woff[w & 1], lds0 + (unsigned)(t % C::W_NST) * W_TILE_BYTES + (cv * 8 + w) * 1024u);
  };
  auto copy_x = [&](int t, int x) {
    dma16(xq + (size_t)t * BK, xoff[x], lds0 + C::X_RING_OFF + (unsigned)(t % C::X_NST) * C::X_STAGE_BYTES + (x * 4 + cv) * 1024u);
  };
  auto copy_s = [&](int t, int i) {
    dma4((const uint8_t*)(sx + (size_t)t * sc.in_kb), soff[i],
         lds0 + C::X_RING_OFF + (unsigned)(t % C::X_NST) * C::X_STAGE_BYTES + C::X_STAGE_S_OFF + sbase(i) * 4u);
  };
  // operation i of the copies that step kb issues: each kind runs its ring's depth ahead of its use
  auto issue_op = [&](int kb, int i) {
    if (C::is_w(i)) copy_w(kb + C::W_PRE, C::w_index(i));
    else if (C::is_s(i)) copy_s(kb + C::X_PRE, C::s_index(i));
    else copy_x(kb + C::X_PRE, C::x_index(i));
  };
  // The item's weight block scales and the flags.  In front of the first copies, in their own order: a load behind them would be waited
  // for with all of them, where the first step needs its own stage alone.
  volatile int* early_flag = (volatile int*)(lds + CLS_FLAG_OFF);
  if (C::W_EARLY && tid < 4) early_flag[tid] = 0;
  const unsigned my_flag = lds0 + CLS_FLAG_OFF + wi * 4;
  const float* wscale = (const float*)(lds + CLS_WSCALE_OFF);   // [2][MAX_KB]
  if (wave < 2) {
    const float* from = MODE == MODE_GATEUP ? (wave ? sw1 : sw0) + ((size_t)e * (N / 128) + item.col_block) * KB
                                            : sw0 + ((size_t)e * (N / 128) + min(item.col_block * 2 + wave, N / 128 - 1)) * KB;
    for (int kk = 0; kk < KB; kk += 64)
      dma4((const uint8_t*)from, (unsigned)min(kk + lane, KB - 1) * 4u, lds0 + CLS_WSCALE_OFF + (wave * MAX_KB + kk) * 4u);
  }
  if (xj == 0) {
    // what the steps before the first would have issued, in their order (completion is counted in issue order)
#pragma unroll
    for (int j = -C::W_PRE; j < 0; ++j) {
#pragma unroll
      for (int i = 0; i < C::OPS; ++i) {
        const int t = j + (C::is_w(i) ? C::W_PRE : C::X_PRE);
        if (t >= 0 && t < KB) issue_op(j, i);
      }
    }
  }

  const float* ws0 = wscale + (MODE == MODE_GATEUP ? 0 : (wi >> 1) * MAX_KB);
  const float* ws1 = wscale + MAX_KB;   // GATEUP only
  wait_lgkm0();   // (the flags are there when the first step's barrier is passed)

  const int lane_off0 = fr * BK + ((fq ^ (fr >> 1)) << 4);         // K bytes [16 fq, +16)
  const int lane_off1 = fr * BK + (((fq + 4) ^ (fr >> 1)) << 4);   // K bytes [64 + 16 fq, +16)
  int wfrag_off[4];
#pragma unroll
  for (int f = 0; f < 4; ++f)
    wfrag_off[f] = (MODE == MODE_GATEUP ? ((f >> 1) * 128 + wi * 32 + (f & 1) * 16) : (wi * 64 + f * 16)) * BK;
  auto read_frag = [&](const uint8_t* base) {
    const v4i lo = *(const v4i*)(base + lane_off0);
    const v4i hi = *(const v4i*)(base + lane_off1);
    return (v8i){lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
  };

  v4f acc[4][XF];
#pragma unroll
  for (int f = 0; f < 4; ++f)
#pragma unroll
    for (int j = 0; j < XF; ++j) acc[f][j] = (v4f){0.f, 0.f, 0.f, 0.f};
  v8i wf[4];
  v4f p[C::NP];
  float pc0 = 0.f, pc1 = 0.f;   // scales of the group whose FMAs are pending
  auto fm = [&](int f, int jj, float c0, float c1) {
    acc[f][jj] += p[(4 * jj + f) % C::NP] * ((MODE == MODE_GATEUP && f >= 2) ? c1 : c0);
  };
  auto mm = [&](int f, int jj, const v8i& x) {
    p[(4 * jj + f) % C::NP] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[f], x, (v4f){0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
  };
  auto fence = [&]() {
    __builtin_amdgcn_sched_barrier(0);
  };
  // group j's MFMAs, each behind the FMAs that finish the one NP before it, and the FMAs still pending behind a step's last group
  auto group = [&](int j, bool pending, const v8i& x, float c0, float c1) {
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      if (f >= C::NP) fm(f - C::NP, j, c0, c1);
      else if (pending) fm(f + 4 - C::NP, j - 1, pc0, pc1);
      mm(f, j, x);
    }
  };
  auto finish = [&]() {
#pragma unroll
    for (int f = 4 - C::NP; f < 4; ++f) fm(f, XF - 1, pc0, pc1);
  };
  // The two waves of a SIMD belong to different wave sets (xj = 0 / 1).  Set 1 runs ROT groups behind set 0: it
  // carries the last ROT activation fragments of a step (and their scales) in registers across the barrier and
  // multiplies them, against the previous step's weights, first thing behind it -- so one wave of each SIMD has
  // matrix work in registers while the other waits for its first fragments from LDS.
  auto run = [&](auto rot_c, auto issue_c) {
    constexpr int ROT = decltype(rot_c)::value;
    constexpr bool ISSUE = decltype(issue_c)::value;   // this wave set issues the copies (and waits for them)
    constexpr int NG = XF - ROT;   // groups of the current step done before the next barrier
    constexpr int NH = ROT > 0 ? ROT : 1;
    v8i held[NH];
    float hc0[NH], hc1[NH];
    // copy_c: what the step issues -- 2: every copy; 1: the activation tile and scales only (the deeper weight
    // ring has reached the item's last K block); 0: nothing
    auto step = [&](int kb, auto first_c, auto copy_c) {
      constexpr bool FIRST = decltype(first_c)::value;
      constexpr int KIND = decltype(copy_c)::value;
      constexpr bool COPY = KIND > 0 && ISSUE;
      constexpr int NOPS = KIND == 2 ? C::OPS : C::XS_OPS;   // (KIND 1 exists only where the activation copies come first)
      // stage kb of both rings has landed once only the copies of later steps are outstanding
      if (!ISSUE) {
        // (the copying waves wait for their copies before the barrier; this set has none in flight)
      } else if (KIND == 2) {
        wait_vm<C::IN_FLIGHT>();
      } else {
        const int rem = KB - 1 - kb;        // the last steps: fewer and fewer copies are in flight
        static_assert(C::W_PRE <= 3, "steps that issue no weight copies are less than W_PRE from the end");
        if (rem >= 2) wait_vm<C::allowed(2)>();
        else if (rem == 1) wait_vm<C::allowed(1)>();
        else wait_vm<0>();
      }
      if (ROT > 0) wait_lgkm0();      // this wave's reads of stage kb - 1 are done before anyone overwrites it
      __builtin_amdgcn_s_barrier();   // stage kb is complete for every wave; every wave is done with stage kb - 1
      if constexpr (ROT > 0) {        // groups NG .. XF-1 of the previous step: held fragments, the previous weights
        if (!FIRST) {
#pragma unroll
          for (int i = 0; i < ROT; ++i) {
            group(NG + i, true, held[i], hc0[i], hc1[i]);
            pc0 = hc0[i];
            pc1 = hc1[i];
            if (COPY) {
#pragma unroll
              for (int o = C::first(i); o < C::first(i + 1); ++o)
                if (o < NOPS) issue_op(kb, o);
            }
            fence();
          }
        } else if (COPY) {
#pragma unroll
          for (int o = 0; o < C::first(ROT); ++o)
            if (o < NOPS) issue_op(kb, o);
        }
      }
      const uint8_t* wt = lds + (kb % C::W_NST) * W_TILE_BYTES;
      const uint8_t* xs = lds + C::X_RING_OFF + (kb % C::X_NST) * C::X_STAGE_BYTES;
      float s0 = ws0[kb], s1 = MODE == MODE_GATEUP ? ws1[kb] : s0;
      if (C::NP < 4) {   // (in scalar registers)
        s0 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(s0)));
        s1 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(s1)));
      }
      const uint8_t* xt = xs + xj * 16 * BK;
      // Every wave of a wave set asks LDS for its first fragments at this moment: the reads come back in issue
      // order, so the first MFMA's operands (activation fragment 0, weight fragment 0) are asked for first and the
      // scales last; the FMAs that finish the previous step's last group run while the reads travel.
      v8i xf[2];
      xf[0] = read_frag(xt);
#pragma unroll
      for (int f = 0; f < 4; ++f) wf[f] = read_frag(wt + wfrag_off[f]);
      float sxv[XF];
      const uint8_t* sp = xs + C::X_STAGE_S_OFF + xj * HALF * 4 + fr * XF * 4;
      {
        if constexpr (C::S_LATE) {
          sxv[0] = *(const float*)sp;
        } else if constexpr (XF % 4 == 0) {
#pragma unroll
          for (int j = 0; j < XF; j += 4) {
            const v4f a = *(const v4f*)(sp + j * 4);
            sxv[j] = a[0]; sxv[j + 1] = a[1]; sxv[j + 2] = a[2]; sxv[j + 3] = a[3];
          }
        } else if constexpr (XF % 2 == 0) {
#pragma unroll
          for (int j = 0; j < XF; j += 2) {
            const float2 a = *(const float2*)(sp + j * 4);
            sxv[j] = a.x; sxv[j + 1] = a.y;
          }
        } else {
#pragma unroll
          for (int j = 0; j < XF; ++j) sxv[j] = *(const float*)(sp + j * 4);
        }
      }
      if (!FIRST) finish();
      fence();
#pragma unroll
      for (int j = 0; j < NG; ++j) {
        if (j + 1 < NG) {
          xf[(j + 1) & 1] = read_frag(xt + (j + 1) * 32 * BK);
          if (C::S_LATE) sxv[j + 1] = *(const float*)(sp + (j + 1) * 4);
        }
        if (ROT > 0 && j == 0) {
#pragma unroll
          for (int i = 0; i < ROT; ++i) {
            if (C::S_LATE) sxv[NG + i] = *(const float*)(sp + (NG + i) * 4);
            held[i] = read_frag(xt + (NG + i) * 32 * BK);
            hc0[i] = sxv[NG + i] * s0;
            hc1[i] = sxv[NG + i] * s1;
          }
        }
        float c0 = 0.f, c1 = 0.f;
        if (C::NP < 4) c0 = sxv[j] * s0, c1 = sxv[j] * s1;
        group(j, j > 0, xf[j & 1], c0, c1);
        // pinned order: the next group's fragment reads first (a whole group of latency cover), then FMA quadruple f
        // just before MFMA f (left alone the compiler puts all 16 FMAs before the 4 MFMAs: down GEMM 3-6 % slower)
        if (j + 1 < NG) __builtin_amdgcn_sched_group_barrier(0x100, C::S_LATE ? 3 : 2, 0);
        if (ROT > 0 && j == 0) {
#pragma unroll
          for (int i = 0; i < ROT; ++i) __builtin_amdgcn_sched_group_barrier(0x100, C::S_LATE ? 3 : 2, 0);
        }
#pragma unroll
        for (int f = 0; f < 4; ++f) {
          if (j > 0 || f >= C::NP) __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
        pc0 = C::NP < 4 ? c0 : sxv[j] * s0;
        pc1 = C::NP < 4 ? c1 : sxv[j] * s1;
        if (C::W_EARLY && COPY && KIND == 2 && ROT + j == C::EARLY_G) {
          // The weight copies from here on overwrite the stage that this step reads: this wave is past its own
          // fragment loads; the other reader of its rows, wave (wi, 1), says so through early_flag.  (It entered the
          // step through the same barrier and signals without waiting for anyone: the loop ends.  Inline assembly
          // so that the unrolled step stays one block for the scheduler.)
          fence();
          int seen;
          asm volatile("1:\n\tds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)\n\tv_cmp_ge_i32 vcc, %2, %0\n\ts_cbranch_vccnz 1b"
                       : "=&v"(seen) : "v"(my_flag), "s"(kb) : "vcc", "memory");
          fence();
        }
        if (COPY) {
#pragma unroll
          for (int o = C::first(ROT + j); o < C::first(ROT + j + 1); ++o)
            if (o < NOPS) issue_op(kb, o);
        }
        fence();
        if (C::W_EARLY && !ISSUE && j == 0) {
          // behind the MFMAs of the first group with this step's weights: all four weight fragments are in registers
          early_flag[wi] = kb + 1;   // (every lane, one value: no branch)
          fence();
        }
      }
    };
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    constexpr std::integral_constant<int, 2> all{};
    constexpr std::integral_constant<int, 1> x_only{};
    constexpr std::integral_constant<int, 0> none{};
    const int n_all = KB - C::W_PRE;   // steps 0 .. n_all-1 issue every copy
    const int n_x = KB - C::X_PRE;     // steps up to n_x-1 still issue the activation tile of a later step
    if (n_all > 0) {
      step(0, yes, all);
    } else {
      bool done = false;
      if constexpr (C::X_FIRST) {
        if (n_x > 0) {
          step(0, yes, x_only);
          done = true;
        }
      }
      if (!done) step(0, yes, none);
    }
    int kb = 1;
    for (; kb < n_all; ++kb) step(kb, no, all);
    if constexpr (C::X_FIRST) {
      for (; kb < n_x; ++kb) step(kb, no, x_only);
    }
    for (; kb < KB; ++kb) step(kb, no, none);
    if constexpr (ROT > 0) {   // the groups carried out of the last step
#pragma unroll
      for (int i = 0; i < ROT; ++i) {
        group(NG + i, true, held[i], hc0[i], hc1[i]);
        pc0 = hc0[i];
        pc1 = hc1[i];
      }
    }
    finish();
  };
  // (fewer groups than that: what there is, or what the register file has room for)
  constexpr int ROT1 = XF >= 10 ? 0 : XF == 9 ? 1 : XF > ROTC ? ROTC : XF - 1;
  if (xj == 0) run(std::integral_constant<int, 0>{}, std::true_type{});
  else run(std::integral_constant<int, ROT1>{}, std::false_type{});
  __syncthreads();   // every wave is done reading the ring before the epilogue reuses LDS

  item_epilogue<MODE, 4, XF, BM, 32, NT, LISTED>(acc, item, xj * 16 + fr, wi, lds, N, out, out_scale, sc, listed);
}

// row tiles of an expert up to which its weight lines are marked non-temporal (grouped_gemm_kernel)
__host__ __device__ inline int once_tiles(int K) { return K <= 2048 ? 2 : 1; }

// The first dense_blocks workgroups serve `dense`, one group of dense_rows rows (the shared expert), whose work items
// follow from the row count alone; the rest serve the routed experts through the work list (hdr null: none).  A
// decode-sized layer runs both in one launch: the shared expert's items are few and as long as the others', and the
// launches, the second stream and the events between them cost it more than the arithmetic.  DENSE false: routed
// items only, as a kernel of its own, because choosing between the two operand sets costs every item of a large
// launch some 0.7 us (0.8 % of the prefill step).
// STREAM: weights come from memory and most experts have one row tile, so items mark their weight lines non-temporal
// where that pays.  Otherwise every copy is a plain one (launch()).
// TALL: tiles of up to 320 rows (moe_tile_rows_voted); a kernel of its own, as the tenth class costs the others 0.5 to 1.5 %.
template <int MODE, bool DENSE, bool STREAM, bool TALL>
__global__ __launch_bounds__(NT, 1) void grouped_gemm_kernel(const GemmOperands routed, TileHeader* hdr,
                                                            const TileEntry* __restrict__ tiles, const GemmOperands dense,
                                                            int dense_rows, int dense_tiles, int dense_blocks) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const bool is_dense = DENSE && (int)blockIdx.x < dense_blocks;   // (dense_blocks is a multiple of 8: the XCD is blockIdx % 8 for both)
  const int K = is_dense ? dense.K : routed.K, N = is_dense ? dense.N : routed.N;
  Item item;
  if (!work_item<MODE, DENSE>(item, lds, N, is_dense, hdr, tiles, dense_rows, dense_tiles, dense_blocks)) return;
  const uint8_t* xq = is_dense ? dense.xq : routed.xq;
  const float* sx = is_dense ? dense.sx : routed.sx;
  const int32_t* row_ids = is_dense ? nullptr : routed.row_ids;
  const uint8_t* w0 = is_dense ? dense.w0 : routed.w0;
  const float* sw0 = is_dense ? dense.sw0 : routed.sw0;
  const uint8_t* w1 = is_dense ? dense.w1 : routed.w1;
  const float* sw1 = is_dense ? dense.sw1 : routed.sw1;
  void* out = is_dense ? dense.out : routed.out;
  float* out_scale = is_dense ? dense.out_scale : routed.out_scale;
  const GemmScales sc = is_dense ? dense.sc : routed.sc;
  const int rows = __builtin_amdgcn_readfirstlane(item.row_count);
#define MOE_ITEM(XF, ONCE) item_body<MODE, XF, ONCE>(item, lds, xq, sx, row_ids, w0, sw0, w1, sw1, K, N, out, out_scale, sc)
  if constexpr (STREAM) {
    // Two row tiles of an expert read the same weight lines; over a short K they stay close enough to find them in L2
    // (non-temporal lines leave it first), over a long one the later tile needs the memory-side cache.  Qwen3-MoE, 4096
    // tokens (K = 2048, 768): 269 us with one-tile experts alone marked, 261 with two; DeepSeek-V3 gate/up (K = 7168) at
    // 4096 tokens: 2426 / 2438 us of the step; all experts whatever their tiles: 8192 tokens 3731 / 3946 us.
    //   Tiles of up to 128 rows are always marked: without a second K loop each the tall classes are 0.1 to 0.3 % faster (shard
    // of 16384 rows 786 / 788 us, Qwen3-MoE of 4096 tokens 267 / 268), and where the lists are short most experts have one
    // tile.  An uneven batch pays for it, as an expert cut into several short tiles is marked too (so / by the rule, normal
    // offsets of 1 to 3 on the logits): full layer, 500 tokens 604 / 602, 394 / 385, 269 / 262 and 211 / 205 us; DeepSeek-V3, 192
    // tokens 1102 / 1097, 467 / 443 and 320 / 315, 256 1055 / 1053, 618 / 601 and 343 / 343, 384 1095 / 1084, 556 / 560 and 543 /
    // 550, 512 1253 / 1256, 682 / 690 and 427 / 430.
    const bool once = __builtin_amdgcn_readfirstlane(item.tiles) <= once_tiles(K);
#define MOE_CLASS(XF) if (once) MOE_ITEM(XF, true); else MOE_ITEM(XF, false); break
    switch ((rows + 31) >> 5) {
      case 10: if constexpr (TALL) { MOE_CLASS(10); }
      case 9: MOE_CLASS(9);
      case 8: MOE_CLASS(8);
      case 7: MOE_CLASS(7);
      case 6: MOE_CLASS(6);
      case 5: MOE_CLASS(5);
      case 4: MOE_ITEM(4, true); break;
      case 3: MOE_ITEM(3, true); break;
      case 2: MOE_ITEM(2, true); break;
      default: MOE_ITEM(1, true); break;
    }
#undef MOE_CLASS
  } else {
    switch ((rows + 31) >> 5) {
      case 10: if constexpr (TALL) { MOE_ITEM(10, false); break; }
      case 9: MOE_ITEM(9, false); break;
      case 8: MOE_ITEM(8, false); break;
      case 7: MOE_ITEM(7, false); break;
      case 6: MOE_ITEM(6, false); break;
      case 5: MOE_ITEM(5, false); break;
      case 4: MOE_ITEM(4, false); break;
      case 3: MOE_ITEM(3, false); break;
      case 2: MOE_ITEM(2, false); break;
      default: MOE_ITEM(1, false); break;
    }
  }
#undef MOE_ITEM
}

// ---- a small layer's batch, straight from the selection ----------------------------------------------------------
//
// Up to 2048 selections of up to 64 experts are read and counted by every workgroup itself, while it would otherwise wait for the
// list header, the list entry and the row ids one after the other: no sort and no list in front of the two GEMMs, and rows of h
// and y stand where their selections stand (flat index token * k + slot).  The same bits; the items too, except where a list could
// have tiles of more than 128 rows, and that an expert's neighbours in the list are others.
//   What bounds these launches: their start (arguments, instruction lines, the selections from memory), then the items' streams as in
// the class kernel.  A GEMM launch is 0.5 to 1.5 us longer than one that reads a list, the sort's launch of 3.5 to 6 us (and as much
// on the host) is gone: tiny layer, 32 tokens 22.6 -> 20 us, 256 25 -> 21.5, 1000 31 -> 28; mini layer, 64 tokens 30 -> 26.5, its
// sublayer 200 tokens 31.6 -> 27.9, 1000 39 -> 35.  Uneven routings (with a list / this way, us a call): normal offsets of 2 on the
// logits, 64 experts of 1024 x 512, k = 8, 200 tokens 46.2 / 35.7, 256 49.0 / 35.1, mini layer of 1024 36.4 / 32.1, tiny of 1000 32.2 /
// 29.6; all 2048 selections of 64 experts at one 46.2 / 36.6, half of 2048 of 32 experts of 1024 x 1024 at one 61.7 / 51.1.  Not every
// one: where an even routing's items just fill the CUs and a few heavy experts begin another round, a list balances that better (the
// 64 experts, 70 % of 200 tokens at eight of them, anywhere 44.9 / 47.8, side by side 46.8 / 42.1; 70 % of 2048 at one 52.0 / 57.7);
// eight experts of 1024 x 2048, 1900 and 2048 rows, 47.7 / 48.5 and 48.9 / 49.8.  The limits are what a lane an expert and four
// selections a thread hold.
constexpr int kScanRows = 2048, kScanExperts = 64, kScanTileRows = 128;
constexpr int SCAN_OFF = 150016;   // LDS: [64] experts' rows, [8] waves' rows of the item's expert, [128] the tile's rows
constexpr int scan_ring() { return cmax(cmax(Cls<1>::RING_BYTES, Cls<2>::RING_BYTES), cmax(Cls<3>::RING_BYTES, Cls<4>::RING_BYTES)); }
static_assert(scan_ring() <= SCAN_OFF && kScanTileRows * 512 <= SCAN_OFF && SCAN_OFF + (kScanExperts + NWAVES + kScanTileRows) * 4 <= CLS_RING, "LDS");

// The workgroup's item among those of the routed rows (false: none is left) and its rows in listed.  MOST: selections of a thread at
// most.  (Few instructions count for more here than few cycles, as every line of them is fetched cold: counts by ballots of the
// selections' bits, with no atomics and two barriers fewer, take 1 to 2 us longer.)
template <int MOST>
__device__ __forceinline__ bool scan_item(Item& item, int* experts, int* counts, int* listed, const int32_t* __restrict__ ids, int R, int E,
                                          int tile_rows, int ncb, int index) {
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), xcd = index & 7;
  const int f = w * MOST * 64 + lane;   // the wave's selections: a run of 64 MOST
  int mine[MOST];
#pragma unroll
  for (int j = 0; j < MOST; ++j) mine[j] = f + 64 * j < R ? ids[f + 64 * j] : -1;
  if (tid < kScanExperts) experts[tid] = 0;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < MOST; ++j)
    if ((unsigned)mine[j] < (unsigned)E) atomicAdd(&experts[mine[j]], 1);   // (a selection out of range has no row)
  __syncthreads();
  // Experts side by side are eight lanes apart: the tiles of a heavy group of them go to all XCDs (of eight that have 70 % of the
  // tokens, 64 experts of 1024 x 512, k = 8, 200 tokens 50.6 -> 42.1 us, 256 51.7 -> 42.2; 46.8 and 52.8 with a list).
  auto swapped = [](int l) { return (l & 7) << 3 | l >> 3; };   // a lane's expert, an expert's lane
  const int rows = experts[swapped(lane)], nt = moe_tile_count(rows, tile_rows), to = moe_wave_scan(nt);
  const int n_items = __builtin_amdgcn_readlane(to, 63) * ncb;
  const int id = (int)((unsigned)(n_items * xcd) >> 3) + (index >> 3);
  if (id >= (int)((unsigned)(n_items * (xcd + 1)) >> 3)) return false;   // (uniform)
  const int tile = id / ncb, at = (int)__builtin_ctzll(__ballot(to > tile)), e = swapped(at);
  const int e_rows = __builtin_amdgcn_readlane(rows, at), e_tiles = __builtin_amdgcn_readlane(nt, at);
  const int first = __builtin_amdgcn_readlane(to, at) - e_tiles;
  int rt, t0;
  expert_item(id - first * ncb, e_tiles, ncb, item.col_block, rt);
  moe_tile_span(e_rows, e_tiles, rt, t0, item.row_count);
  item.expert = e;
  item.tiles = e_tiles;
  item.row_start = 0;
  unsigned long long here[MOST];
  int count = 0;
#pragma unroll
  for (int j = 0; j < MOST; ++j) {
    here[j] = __ballot(mine[j] == e);
    count += __popcll(here[j]);
  }
  if (lane == 0) counts[w] = count;
  __syncthreads();
  int place = -t0;   // in the tile, of the wave's first row
  for (int v = 0; v < w; ++v) place += counts[v];
#pragma unroll
  for (int j = 0; j < MOST; ++j) {
    const int p = place + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(here[j] >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)here[j], 0u));
    if (mine[j] == e && (unsigned)p < (unsigned)item.row_count) listed[p] = f + 64 * j;
    place += __popcll(here[j]);
  }
  __syncthreads();
  return true;
}

template <int MODE, bool DENSE, int MOST>
__global__ __launch_bounds__(NT, 1) void scan_gemm_kernel(const GemmOperands routed, const int32_t* __restrict__ ids, int R, int E, int k,
                                                         int tile_rows, const GemmOperands dense, int dense_rows, int dense_tiles,
                                                         int dense_blocks) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  int* const experts = (int*)(lds + SCAN_OFF);
  int* const counts = experts + kScanExperts;
  int* const listed = counts + NWAVES;
  const bool is_dense = DENSE && (int)blockIdx.x < dense_blocks;
  const GemmOperands op = is_dense ? dense : routed;
  const int ncb = MODE == MODE_GATEUP ? op.N / 128 : (op.N + 255) / 256;
  Item item;
  if (is_dense) {
    if (!work_item<MODE, true>(item, lds, op.N, true, nullptr, nullptr, dense_rows, dense_tiles, dense_blocks)) return;
    if ((int)threadIdx.x < item.row_count) listed[threadIdx.x] = item.row_start + threadIdx.x;
    __syncthreads();
  } else if (!scan_item<MOST>(item, experts, counts, listed, ids, R, E, tile_rows, ncb, (int)blockIdx.x - (DENSE ? dense_blocks : 0))) {
    return;
  }
  const int div = MODE == MODE_GATEUP && !is_dense ? k : 1;
#define MOE_ITEM(XF) item_body<MODE, XF, false, true>(item, lds, op.xq, op.sx, nullptr, op.w0, op.sw0, op.w1, op.sw1, op.K, op.N, op.out, op.out_scale, op.sc, listed, div)
  switch ((__builtin_amdgcn_readfirstlane(item.row_count) + 31) >> 5) {
    case 4: MOE_ITEM(4); break;
    case 3: MOE_ITEM(3); break;
    case 2: MOE_ITEM(2); break;
    default: MOE_ITEM(1); break;
  }
#undef MOE_ITEM
}

int col_blocks(int mode, int N) { return mode == MODE_GATEUP ? N / 128 : (N + 255) / 256; }

int max_tiles_for(int R, int E, int tile_rows) { return (int)(((long long)R + tile_rows - 1) / tile_rows + (E < R ? E : R)); }
// fewest work items at which every launch takes full tiles (moe_gemm_tile_rows)
constexpr int kFullTileItems = 768;

// Lists whose pool may be large: of up to 8 rounds at most (the fewer, the larger a part the last one is; up to 10 the
// expert-parallel shard of 16384 rows takes 786 us, up to 8 778), of items of 12 K steps (14 us) and more.  Shorter items lose
// more by the draw (Qwen3-MoE, 2800 tokens 217 -> 221 us, 4000 of the mini layer 76 -> 79.5).
//   32 experts of 7168 x 2048, all or 29 of them with rows, Zipf(0.8 / 1.2 / 1.6), 560 to 3600 rows in 80s, large pool against small:
// gate/up -6.3 % on average (-28 % where the last round came out worst), down -4.0 %; up to 10000 rows alike.  Not for lists of one
// or two full rounds of items (moe_tile_first): equal shares end together there and draws do not (2000 to 2240 rows, 32 tiles of 16
// columns: 154 to 173 us, 176 to 184 with the large pool; else +0.6 to +4.5 %).  It still loses now and then where the shares
// nearly are whole rounds (31 tiles, 1200 to 1440 rows of Zipf(1.6): +5 to +13 %; other 31 tiles -1 to -11 %).
int moe_gemm_pool_tiles(int max_tiles, int tile_rows, int ncb_least, int kb) {
  const bool few = (long long)max_tiles * ncb_least <= 8 * 256 && kb >= 12 && tile_rows > kStreamRows;
  return few ? max_tiles >> 2 : max_tiles >> 4;
}

// ncb: column blocks of the list's GEMMs (0: none); kb: the fewest K steps of these
TileList tile_list(void* ws, int R, int E, int tile_rows, int ncb_gateup, int ncb_down, int kb) {
  const int max_tiles = max_tiles_for(R, E, tile_rows < kTileRows ? tile_rows : kTileRows), ncb = ncb_down && ncb_down < ncb_gateup ? ncb_down : ncb_gateup;
  return TileList{max_tiles, moe_gemm_pool_tiles(max_tiles, tile_rows, ncb, kb), R, tile_rows, (TileHeader*)ws,
                  (TileEntry*)((char*)ws + sizeof(TileHeader)), {ncb_gateup, ncb_down},
                  {(32 << kTileQBits) / (ncb_gateup ? ncb_gateup : 1), (32 << kTileQBits) / (ncb_down ? ncb_down : 1)}};
}

int check_operands(const GemmOperands& op, int rows, int E, int mode, const char* what) {
  MOE_REQUIRE((rows == 0 || (op.xq && op.sx && op.out && (mode == MODE_DOWN || op.out_scale))) && op.w0 && op.sw0 &&
                  (mode == MODE_DOWN || (op.w1 && op.sw1)), MOE_ERR_NULL, "%s: null pointer", what);
  MOE_REQUIRE(E >= 1 && E <= 1024 && rows >= 0 && op.K > 0 && op.N > 0 && op.K % 128 == 0 && op.N % 128 == 0, MOE_ERR_BAD_SHAPE,
              "%s: need contraction and output sizes in multiples of 128 and 1 <= E <= 1024, got E=%d rows=%d K=%d N=%d", what, E,
              rows, op.K, op.N);
  MOE_REQUIRE(MOE_ALIGNED16(op.xq) && MOE_ALIGNED16(op.w0) && MOE_ALIGNED16(op.w1) && MOE_ALIGNED16(op.out), MOE_ERR_BAD_ALIGN,
              "%s: pointers must be 16-byte aligned", what);
  MOE_REQUIRE((long long)rows * op.sc.in_row * 4 <= (1ll << 32) &&
                  (mode == MODE_DOWN || (long long)rows * op.sc.out_row + (long long)(op.N / 128) * op.sc.out_cb <= (1ll << 40)),
              MOE_ERR_BAD_SHAPE, "%s: scale array out of the addressable range", what);
  MOE_REQUIRE(op.K <= MAX_KB * BK, MOE_ERR_BAD_SHAPE, "%s: contraction length %d exceeds %d", what, op.K, MAX_KB * BK);
  MOE_REQUIRE((long long)op.N * op.K <= (1ll << 32) && (long long)rows * op.K <= (1ll << 32), MOE_ERR_BAD_SHAPE,
              "%s: one expert matrix and the activation array must each stay within 4 GB (N=%d K=%d rows=%d)", what, op.N, op.K, rows);
  return MOE_OK;
}

}  // namespace

int moe_gemm_check(const GemmOperands& op, int rows, int E, bool down) {
  return check_operands(op, rows, E, down ? MODE_DOWN : MODE_GATEUP, down ? "gemm_down" : "gemm_gateup");
}
namespace {

template <int MODE>
int launch(const RoutedGemm* rt, const DenseGemm* dn, hipStream_t s) {
  const char* what = MODE == MODE_GATEUP ? "gemm_gateup" : "gemm_down";
  // A launch of short tiles is a weight stream, and writes in between cost the HBM far more than their bytes (512
  // experts of 40 rows, down GEMM of K = 1024: 416 us with plain stores, 345 with none, at 6 % of the bytes).  Written
  // through at once they cost half of that (380 us): DeepSeek-V3, 777 tokens 1395 -> 1370 us; full layer, 4096 tokens
  // 1420 -> 1387.  An output that the L2s can keep until its reader comes stays there, and a launch of taller tiles
  // has other limits (Qwen3-MoE, 2000 tokens = 125 rows an expert: 195 us plain, 200 through).
  auto through = [](int rows, int E, int N) {
    return (size_t)rows * N * (MODE == MODE_DOWN ? 2 : 1) > ((size_t)4 << 20) && rows <= 96ll * E;
  };
  auto own_tile_rows = [](int rows, int E, const GemmOperands& op) {
    TileShape t{rows, E, rows, {0, 0}, {0, 0}, 0, {0, 0}};
    t.ncb[MODE] = col_blocks(MODE, op.N), t.kb[MODE] = op.K / BK;
    return moe_gemm_tile_rows(t);
  };
  GemmOperands routed{}, dense{};
  TileList l{};
  int dense_rows = 0, dense_tiles = 0, dense_tile_rows = 0;
  long long dense_blocks = 0, grid = 0;
  if (dn) {
    // (both groups in one launch are cut alike: it goes to one kernel by the height of one list's tiles)
    MOE_REQUIRE(!rt || rt->list_tile_rows, MOE_ERR_BAD_SHAPE, "%s: a dense group beside routed rows needs their list to be there", what);
    if (int rc = check_operands(dn->op, dn->rows, 1, MODE, what)) return rc;
    dense = dn->op;
    dense.sc.out_through = through(dn->rows, 1, dense.N);
    dense_rows = dn->rows;
    dense_tile_rows = rt ? rt->list_tile_rows : own_tile_rows(dense_rows, 1, dense);
    dense_tiles = moe_tile_count(dense_rows, dense_tile_rows);
    dense_blocks = 8 * (((long long)dense_tiles * col_blocks(MODE, dense.N) + 7) / 8);
    grid = dense_blocks;
  }
  if (rt && rt->ids) {   // (moe_gemm_scan_rows)
    if (int rc = check_operands(rt->op, rt->R, rt->E, MODE, what)) return rc;
    routed = rt->op;
    routed.sc.out_through = through(rt->R, rt->E, routed.N);
    grid += 8 * (((long long)max_tiles_for(rt->R, rt->E, rt->list_tile_rows) * col_blocks(MODE, routed.N) + 7) / 8);
    static std::atomic<unsigned long long> lds_raised[6] = {};
    const int most = rt->R <= NT ? 0 : rt->R <= 2 * NT ? 1 : 2;
    auto* kernel = most == 0 ? (dn ? scan_gemm_kernel<MODE, true, 1> : scan_gemm_kernel<MODE, false, 1>)
                 : most == 1 ? (dn ? scan_gemm_kernel<MODE, true, 2> : scan_gemm_kernel<MODE, false, 2>)
                             : (dn ? scan_gemm_kernel<MODE, true, kScanRows / NT> : scan_gemm_kernel<MODE, false, kScanRows / NT>);
    if (int rc = moe_raise_lds_limit((const void*)kernel, CLS_LDS_BYTES, lds_raised[2 * most + (dn != nullptr)])) return rc;
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(NT), CLS_LDS_BYTES, s, routed, rt->ids, rt->R, rt->E, rt->k, rt->list_tile_rows,
                       dense, dense_rows, dense_tiles, (int)dense_blocks);
    return moe_check_hip(hipGetLastError(), "gemm launch");
  }
  if (rt) {
    MOE_REQUIRE(rt->group_offsets && rt->ws, MOE_ERR_NULL, "%s: null pointer", what);
    if (int rc = check_operands(rt->op, rt->R, rt->E, MODE, what)) return rc;
    MOE_REQUIRE(MOE_ALIGNED16(rt->ws), MOE_ERR_BAD_ALIGN, "%s: pointers must be 16-byte aligned", what);
    const size_t need = moe_gemm_workspace_bytes(rt->R, rt->E, rt->op.N);
    MOE_REQUIRE(rt->ws_bytes >= need, MOE_ERR_WORKSPACE_TOO_SMALL, "%s: workspace %zu < %zu", what, rt->ws_bytes, need);
    if (rt->R > 0) {
      routed = rt->op;
      routed.sc.out_through = through(rt->R, rt->E, routed.N);
      l = tile_list(rt->ws, rt->R, rt->E, rt->list_tile_rows ? rt->list_tile_rows : own_tile_rows(rt->R, rt->E, routed),
                    col_blocks(MODE, routed.N), 0, routed.K / BK);   // (one launch reads a list that it builds itself)
      if (rt->list_tile_rows) l.pool_tiles = rt->list_pool_tiles;
      // sized by the worst case of the largest XCD share (moe_xcd_share_cap_q) and of an XCD's draws from the pool;
      // surplus workgroups exit at once
      const long long max_items = (long long)l.max_tiles * col_blocks(MODE, routed.N);
      const long long pool_max = (long long)l.pool_tiles * col_blocks(MODE, routed.N);
      grid += 8 * ((max_items + 7) / 8 + 2 + moe_pool_workgroups(pool_max));
    }
  }
  MOE_REQUIRE(grid < (1ll << 30), MOE_ERR_BAD_SHAPE, "%s: %lld work items exceed the grid limit", what, grid);
  if (grid == 0) return MOE_OK;
  if (l.hdr && !rt->list_tile_rows) {
    const bool wave = rt->E <= MOE_WAVE && !many_tiles_each(rt->E, l.max_tiles);
    hipLaunchKernelGGL(wave ? build_tiles_kernel<true> : build_tiles_kernel<false>, dim3(1), dim3(wave ? MOE_WAVE : 1024), 0, s,
                       rt->group_offsets, rt->E, rt->R, l);
  }
  // Non-temporal weight copies gain a stream from memory 2 to 3 % (four experts of 7168 x 2048 among others, 1 row each:
  // 46.6 -> 45.4 us, 64 tokens of the DeepSeek-V3 layer 12 %) and cost
  //  - a third where the memory-side cache (256 MB) still holds the weights from the call before (the same four experts
  //    over and over 29.3 / 44.9 us; tiny layer, 64 tokens 23.9 / 26.0, 256 25.3 / 27.3; mini sublayer, 64 tokens 36.9 /
  //    39.5, 256 37.8 / 40.6): layers of up to 192 MB, three projections of this size, go without (moe_gemm_from_memory);
  //  - as much where the several short tiles of a small problem's experts read the same lines (four experts of 7168 x 2048
  //    from memory, 40 rows each 49.7 / 55.0 us, 200 51.8 / 60.6; tiny layer, 2048 tokens 48.9 / 52.1).
  const bool from_memory = moe_gemm_from_memory((rt ? 1ll * rt->E * rt->op.N * rt->op.K : 0) + (dn ? 1ll * dn->op.N * dn->op.K : 0));
  const bool shared_lines = l.hdr ? l.tile_rows <= 128 && rt->R > (long long)once_tiles(routed.K) * l.tile_rows * rt->E
                                  : dense_tiles > once_tiles(dense.K) && dense_rows <= 128 * dense_tiles;
  const bool stream = from_memory && !shared_lines;
  const int tallest = l.hdr ? l.tile_rows : dense_tile_rows;   // (a dense group beside routed ones is cut as their list is)
  long long items = dn ? (long long)dense_tiles * col_blocks(MODE, dense.N) : 0;
  if (l.hdr) items += (long long)(rt->E < rt->R ? rt->E : rt->R) * col_blocks(MODE, routed.N);
  if (moe_gemm_streams(MODE, tallest, items))
    return moe_gemm_stream_launch(MODE, StreamLaunch{routed, l.hdr, l.tiles, l.rows, dense, dense_rows, dense_tiles, (int)dense_blocks,
                                                     stream, (unsigned)grid, tallest}, s);
  static std::atomic<unsigned long long> lds_raised[6] = {};
  const bool tall = !dn && tallest > kTileRows;
  auto* kernel = dn ? (stream ? grouped_gemm_kernel<MODE, true, true, false> : grouped_gemm_kernel<MODE, true, false, false>)
               : tall ? (stream ? grouped_gemm_kernel<MODE, false, true, true> : grouped_gemm_kernel<MODE, false, false, true>)
                      : (stream ? grouped_gemm_kernel<MODE, false, true, false> : grouped_gemm_kernel<MODE, false, false, false>);
  const int lds = tall ? TALL_LDS_BYTES : CLS_LDS_BYTES;
  if (int rc = moe_raise_lds_limit((const void*)kernel, lds, lds_raised[(dn ? 2 : tall ? 4 : 0) + stream])) return rc;
  hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(NT), lds, s, routed, l.hdr, l.tiles, dense, dense_rows,
                     dense_tiles, (int)dense_blocks);
  return moe_check_hip(hipGetLastError(), "gemm launch");
}

}  // namespace

// Full tiles where they give every CU several work items; a smaller problem is cut so that its rounds over the 256 CUs
// take the shortest time: a work item costs about (8 + height) per K step, in units of 32 rows, and some 50 of these
// besides (list entry, first copies, epilogue).  8 experts of 64 rows were 16 work items of the down GEMM, on 256 CUs.
// The groups are taken to be two standard deviations of an even routing above their mean, so that a count of tiles
// that just fills a round does not spill into another one.  One group's size is known, and so are its rounds however many
// items they hold: 8192 rows of 2048 x 8192 are 8 rounds of 256-row tiles or of 288-row ones, 287 -> 274 us (gate/up),
// 138.6 -> 127.1 the down GEMM of 7168 x 2048.
//   Before that: short tiles, which moe_gemm_stream.hip takes -- 32 rows, or 128 where a down GEMM reads the list (no gate/up
// launch of these goes there, and on the class kernel it is better off with tall tiles and their larger pool: 264 to 512 rows
// for 32 experts of 7168 x 2048, uneven, -6.5 to +2 %, -1.5 on average) -- where no expert can have more rows, or hardly one
// will, with eight times the mean to spare.  An expert that has more after all is cut, and its weights are read once for each
// tile, from L2 at best.  That is why the lines lie at 4 and 16 rows an expert (4000 tokens of the full layer, 78 rows an
// expert, cut to 128 rows: 1329 us where the routing is even, 1380 for 1340 where 81 experts have 128 to 493).  Below them, against
// the heights by the rounds, routing even or uneven by normal offsets of 1 and 2 on the logits: Qwen3-MoE, 20 tokens 86 / 93, 59 /
// 63, 41 / 42.5 us; 100 tokens 110.7 / 114.5, 84.9 / 84.5, 67.2 / 69.7; 64 tokens 103 / 111, 73.5 / 79.5, but 57.7 / 54.3, where five
// experts of 33 to 52 rows begin another round; 128 tokens of DeepSeek-V3 984 / 994, 644 / 643, 353 / 349; full layer, 100 tokens
// 844 / 855, 400 1037 / 1062, 256 1028 / 1019.  A shared expert beside them is cut alike: where the two tiles that 84 tokens of the
// DeepSeek-V3 layer have more than in one of 96 rows begin another round of items (125 experts touched, which the host does
// not know) 852 / 835; 33 to 128 tokens otherwise -1.0 to +1.5 %, -0.2 on average.
//   Tall tiles (320 rows, moe_tile_rows_voted) for lists of both GEMMs, of short K and at most eight rounds, where an even routing
// puts the largest groups, 2.5 to 3 standard deviations above the mean, between whole full tiles and whole tall ones: with full
// tiles alone a few of Qwen3-MoE's 128 experts have two at 4096 tokens, some 130 tiles x 6 and x 8 columns, 3.05 and 4.06 rounds.  Even
// logits, six draws each, the launches' medians full / tall: 4096 tokens gate/up 134 / 128, down 91 / 84 (of these the two draws that have
// an expert of more than 320 rows, and so full tiles, 146 / 143 and 130 / 135, 96 / 90 and 86 / 87), 8192 226 / 224 and 150 / 145, 9000 250 /
// 236 and 167 / 155; the layer, 4096 tokens 258 / 244, 4300 267 / 256, 9000 482 / 476 and 490 / 474.  For 128 experts, k = 8, that is 3850 to
// 4430 and 8120 to 9240 tokens.  The kernel that has this height too runs the other heights slower, which is what a wrong guess
// costs: the layer with normal offsets of 0.15 to 2 on the logits -1.8 to +0.9 % at 3860 to 4430 tokens, -0.2 to +2 % at 8120 to 9240.  Hence
// only where the guess has shown to be right more often than not: not for rows that another GPU has dispatched, which are uneven,
// nor for longer K, of which one batch was measured (K = 7168, 64 experts of 266 rows each, gate/up 538 / 504, down 298 / 289) and no
// uneven one, nor between 2048 and that.
int moe_gemm_tile_rows(const TileShape& t) {
  const int groups = t.E < t.R ? t.E : t.R;
  if (groups <= 0) return kTileRows;
  if ((t.max_rows <= 32 || t.R <= 4 * t.E) && (long long)groups * (t.ncb[0] > t.ncb[1] ? t.ncb[0] : t.ncb[1]) >= kStreamItems) return 32;
  if ((t.max_rows <= kStreamRows || t.R <= kStreamRows / 8 * t.E) && (long long)groups * t.ncb[1] >= kStreamItems) return kStreamRows;
  const int mean = (t.R + groups - 1) / groups;
  if (mean > kFullTileItems * kTileRows / groups) return kTileRows;
  const int least = !t.ncb[0] || (t.ncb[1] && t.ncb[1] < t.ncb[0]) ? t.ncb[1] : t.ncb[0];
  int spread = 0;
  while (t.E > 1 && spread * spread < 4 * mean) ++spread;
  if (t.E > 1 && groups * ((mean + kTileRows - 1) / kTileRows) * least >= kFullTileItems) {
    const int n = moe_tall_tiles(t.R, t.E), longest = t.kb[0] > t.kb[1] ? t.kb[0] : t.kb[1];
    const bool may_end_alike = 2 * mean + 3 * spread > 2 * n * kTileRows && 4 * mean + 5 * spread <= 4 * n * kTallTileRows;
    return t.ncb[0] && t.ncb[1] && !t.dense_rows && longest <= 16 && (long long)groups * n * least <= 8 * 256 && may_end_alike ? kTallTileRows : kTileRows;
  }
  const int units = (mean + spread + 31) / 32, dense_units = (t.dense_rows + 31) / 32;
  int best = 0, best_u = kTileRows / 32;
  for (int u = kTileRows / 32; u >= 1; --u) {
    const int nt = (units + u - 1) / u, dense_nt = (dense_units + u - 1) / u, tallest = units > dense_units ? units : dense_units, height = tallest < u ? tallest : u;
    int time = 0;
    for (int g = 0; g < 2; ++g)
      time += (groups * nt * t.ncb[g] + dense_nt * t.dense_ncb[g] + 255) / 256 * ((8 + height) * t.kb[g] + (t.kb[g] ? 50 : 0));
    if (best == 0 || time < best) best = time, best_u = u;
  }
  return 32 * best_u;
}

// The two GEMMs want different heights where K of the down GEMM is short: tall tiles for gate/up, and for down 128 rows, which the kernel
// with two workgroups a CU takes (moe_gemm_stream.hip), because start and end are a good part of an item of up to 8 K steps and another
// workgroup works meanwhile.  The placing launch writes both lists, in two workgroups.  The down launch alone, gate/up's list / its own, even
// routing or uneven by normal offsets of 1 and 2 on the logits: Qwen3-MoE (6 K steps), 400 tokens 39.6 / 36.5 us, 1000 47.0 / 41.4, 2000
// 63.0 / 55.6 and 60.4 / 56.8 and 49.2 / 46.2, 3000 71.8 / 64.8; full layer (8), 1000 389 / 367, 2047 405 / 381, 312 / 307 and 188 / 180.
//   The lines (the call, one list / two, routed as above): Qwen3-MoE, 300 tokens 123.4 / 120.0, 109.9 / 105.7 and 76.4 / 74.9, 3000 (188
// rows an expert) 217.5 / 215.9, 231.7 / 221.2 and 218.1 / 206.7, 3800 (238) 241.6 / 245.3, 269.6 / 262.1 and 241.0 / 234.2, 5000 323.9 / 322.7,
// 313.6 / 309.2 and 308.2 / 309.7; full layer, 900 tokens 1046 / 1025, 692 / 678 and 324 / 318, 3000 (59 rows) 1216 / 1200, 1034 /
// 1033 and 668 / 667, 4096 (80) 1315 / 1299, 1191 / 1198 and 879 / 884; DeepSeek-V3 (16 K steps), 777 (24) 1376 / 1378, 1058 / 1082 and
// 519 / 523.  Two lists (and the weights' scales in front of the copies, 1 to 3 %) against one without these, 128 experts of 2048 x 128 to
// 1024 (1 to 8 K steps), k = 8, and others of 512 to 7168 x 256 to 768, 17 to 195 rows an expert, even routing and offsets of 1 and 4: 0.79 to
// 1.02, on average 0.96; above 1.005 at six of 288, four of them with an offset of 4, where a few experts have most rows.
//   A shared expert of long K beside is cut into short tiles too, and one such item can outlast the launch: not where it has more than 16
// K steps, and 7/4 of those that a place (two workgroups a CU) has on average, unless the shared expert is one tall tile or two thirds of
// the routed work.  Qwen3-MoE beside a shared expert of 3072 (24 K steps), 384 tokens 139 / 142 us, 640 151 / 150; of 4096, 384 140 / 150, 640 155 / 161,
// 960 171 / 174; of 6144, 272 189 / 152, 384 151 / 167, 640 172 / 183, 1200 206 / 212, 1440 230 / 223; 256 experts of 1024 x 512 beside
// one of 4096, 640 117 / 122; of 4096 x 512 beside one of 4096, 544 352 / 335.
int moe_gemm_down_tile_rows(const TileShape& t, int list_rows) {
  const int groups = t.E < t.R ? t.E : t.R;
  if (t.R <= kSmallRows || t.R > kFullTileItems * kTileRows || list_rows <= kStreamRows || list_rows > kTileRows) return 0;
  if ((long long)groups * t.ncb[1] < kStreamItems || t.kb[1] > 8 || t.R > (t.kb[1] <= 6 ? 200ll : 64ll) * t.E) return 0;
  const int dense_kb = t.dense_ncb[0];   // (the shared expert's columns in gate/up)
  if (t.dense_rows > list_rows && dense_kb > 16) {
    const long long routed = (long long)groups * t.ncb[1] * t.kb[1], dense = (long long)moe_tile_count(t.dense_rows, kStreamRows) * t.dense_ncb[1] * dense_kb;
    if (4ll * 512 * dense_kb > 7 * (routed + dense) && 3 * dense < 2 * routed) return 0;
  }
  return kStreamRows;
}

// Batches whose GEMMs read the selection themselves: few rows of few experts whose launches are ones of the class kernel with plain
// weight copies and tiles of up to 128 rows (a list's tiles may be allowed more where hardly any expert will have so many).
int moe_gemm_scan_rows(const TileShape& t, bool from_memory) {
  if (t.R < 1 || t.R > kScanRows || t.E > kScanExperts || from_memory) return 0;
  const int groups = t.E < t.R ? t.E : t.R, mean = (t.R + groups - 1) / groups;
  int spread = 0;
  while (spread * spread < 4 * mean) ++spread;
  const int list_rows = moe_gemm_tile_rows(t), rows = list_rows < kScanTileRows ? list_rows : kScanTileRows;
  if (rows < list_rows && mean + spread > kScanTileRows) return 0;
  for (int g = 0; g < 2; ++g)
    if (moe_gemm_streams(g == 0 ? MODE_GATEUP : MODE_DOWN, rows, (long long)groups * t.ncb[g] + (long long)moe_tile_count(t.dense_rows, rows) * t.dense_ncb[g]))
      return 0;
  return rows;
}

extern "C" size_t moe_gemm_workspace_bytes(int R, int E, int N_out) {
  (void)N_out;   // the tile list does not depend on the number of output columns
  // lists of short tiles exist below kFullTileItems full tiles only
  int tiles = max_tiles_for(R, E, kTileRows);
  const int few = R < kFullTileItems * kTileRows ? R : kFullTileItems * kTileRows;
  if (max_tiles_for(few, E, 32) > tiles) tiles = max_tiles_for(few, E, 32);
  return sizeof(TileHeader) + (size_t)tiles * sizeof(TileEntry) + 256;
}

int moe_gemm_gateup_impl(const RoutedGemm* routed, const DenseGemm* dense, moe_stream_t stream) {
  return launch<MODE_GATEUP>(routed, dense, (hipStream_t)stream);
}
int moe_gemm_down_impl(const RoutedGemm* routed, const DenseGemm* dense, moe_stream_t stream) {
  return launch<MODE_DOWN>(routed, dense, (hipStream_t)stream);
}

namespace {
int gateup(const uint8_t* xq, const float* sx, const int32_t* row_ids, const uint8_t* w_gate, const float* sw_gate,
           const uint8_t* w_up, const float* sw_up, const int32_t* group_offsets, int E, int R, int D, int I, uint8_t* hq,
           float* sh, void* ws, size_t ws_bytes, GemmScales sc, moe_stream_t stream) {
  const RoutedGemm r{{xq, sx, row_ids, w_gate, sw_gate, w_up, sw_up, D, I, hq, sh, sc}, group_offsets, E, R, ws, ws_bytes, 0, 0};
  return moe_gemm_gateup_impl(&r, nullptr, stream);
}
int down(const uint8_t* hq, const float* sh, const uint8_t* w_down, const float* sw_down, const int32_t* group_offsets, int E,
         int R, int I, int D, void* y_bf16, void* ws, size_t ws_bytes, GemmScales sc, moe_stream_t stream) {
  const RoutedGemm r{{hq, sh, nullptr, w_down, sw_down, nullptr, nullptr, I, D, y_bf16, nullptr, sc}, group_offsets, E, R, ws,
                     ws_bytes, 0, 0};
  return moe_gemm_down_impl(&r, nullptr, stream);
}
}  // namespace

extern "C" int moe_gemm_gateup_swiglu_fp8(const uint8_t* xq, const float* sx, const int32_t* row_ids,
                                          const uint8_t* w_gate, const float* sw_gate, const uint8_t* w_up,
                                          const float* sw_up, const int32_t* group_offsets, int E, int R, int D,
                                          int I, uint8_t* hq, float* sh, void* ws, size_t ws_bytes,
                                          moe_stream_t stream) {
  return gateup(xq, sx, row_ids, w_gate, sw_gate, w_up, sw_up, group_offsets, E, R, D, I, hq, sh, ws, ws_bytes,
                moe_row_major_scales(D, I), stream);
}

namespace {
int check_layout(int layout, const char* what) {
  MOE_REQUIRE(layout == MOE_SCALES_ROW_MAJOR || layout == MOE_SCALES_BLOCK_MAJOR, MOE_ERR_BAD_SHAPE,
              "%s: unknown scale layout %d", what, layout);
  return MOE_OK;
}
}  // namespace

extern "C" int moe_gemm_gateup_swiglu_fp8_layout(const uint8_t* xq, const float* sx, const int32_t* row_ids,
                                                 const uint8_t* w_gate, const float* sw_gate, const uint8_t* w_up,
                                                 const float* sw_up, const int32_t* group_offsets, int E, int R, int D,
                                                 int I, uint8_t* hq, float* sh, void* ws, size_t ws_bytes, int sx_layout,
                                                 int sh_layout, moe_stream_t stream) {
  if (int rc = check_layout(sx_layout, "gemm_gateup: sx")) return rc;
  if (int rc = check_layout(sh_layout, "gemm_gateup: sh")) return rc;
  GemmScales sc = moe_row_major_scales(D, I);
  if (sx_layout == MOE_SCALES_BLOCK_MAJOR) sc.in_row = 1, sc.in_kb = R, sc.in_listed = true;
  if (sh_layout == MOE_SCALES_BLOCK_MAJOR) sc.out_row = 1, sc.out_cb = R;
  return gateup(xq, sx, row_ids, w_gate, sw_gate, w_up, sw_up, group_offsets, E, R, D, I, hq, sh, ws, ws_bytes, sc, stream);
}

namespace {
// The device address of `scratch` on the current device, looked up once per device.
int static_scratch(void** out) {
  static std::mutex mu;
  static void* ptrs[64] = {};
  int dev = 0;
  if (int rc = moe_check_hip(hipGetDevice(&dev), "static scratch: hipGetDevice")) return rc;
  MOE_REQUIRE(dev >= 0 && dev < 64, MOE_ERR_HIP, "static scratch: device index %d out of range", dev);
  std::lock_guard<std::mutex> lock(mu);
  if (!ptrs[dev]) {
    void* p = nullptr;
    if (int rc = moe_check_hip(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "static scratch: hipGetSymbolAddress")) return rc;
    MOE_REQUIRE(p != nullptr, MOE_ERR_HIP, "static scratch: no device address");
    ptrs[dev] = p;
  }
  *out = ptrs[dev];
  return MOE_OK;
}
}  // namespace

extern "C" int moe_gemm_gateup_swiglu_fp8_static(const uint8_t* xq, const float* sx, const int32_t* row_ids,
                                                 const uint8_t* w_gate, const float* sw_gate, const uint8_t* w_up,
                                                 const float* sw_up, const int32_t* group_offsets, int E, int R,
                                                 int D, int I, uint8_t* hq, float* sh, moe_stream_t stream) {
  MOE_REQUIRE(E >= 1 && E <= 1024 && R >= 0, MOE_ERR_BAD_SHAPE, "gemm_gateup_static: need 1 <= E <= 1024, got E=%d R=%d", E, R);
  const size_t need = moe_gemm_workspace_bytes(R, E, I);
  MOE_REQUIRE(need <= (size_t)MOE_STATIC_SCRATCH_BYTES, MOE_ERR_WORKSPACE_TOO_SMALL,
              "gemm_gateup_static: the tile list of R=%d rows, E=%d experts needs %zu bytes, the static scratch holds %u",
              R, E, need, (unsigned)MOE_STATIC_SCRATCH_BYTES);
  void* ws = nullptr;
  if (int rc = static_scratch(&ws)) return rc;
  // the tile list (header and every entry the GEMM reads) is rewritten by this call's first kernel: nothing of
  // an earlier call's contents is read
  return gateup(xq, sx, row_ids, w_gate, sw_gate, w_up, sw_up, group_offsets, E, R, D, I, hq, sh, ws, MOE_STATIC_SCRATCH_BYTES,
                moe_row_major_scales(D, I), stream);
}

extern "C" int moe_gemm_down_fp8(const uint8_t* hq, const float* sh, const uint8_t* w_down, const float* sw_down,
                                 const int32_t* group_offsets, int E, int R, int I, int D, void* y_bf16, void* ws,
                                 size_t ws_bytes, moe_stream_t stream) {
  return down(hq, sh, w_down, sw_down, group_offsets, E, R, I, D, y_bf16, ws, ws_bytes, moe_row_major_scales(I, D), stream);
}

extern "C" int moe_gemm_down_fp8_layout(const uint8_t* hq, const float* sh, const uint8_t* w_down, const float* sw_down,
                                        const int32_t* group_offsets, int E, int R, int I, int D, void* y_bf16,
                                        void* ws, size_t ws_bytes, int sh_layout, moe_stream_t stream) {
  if (int rc = check_layout(sh_layout, "gemm_down: sh")) return rc;
  GemmScales sc = moe_row_major_scales(I, D);
  if (sh_layout == MOE_SCALES_BLOCK_MAJOR) sc.in_row = 1, sc.in_kb = R, sc.in_listed = true;
  return down(hq, sh, w_down, sw_down, group_offsets, E, R, I, D, y_bf16, ws, ws_bytes, sc, stream);
}

// The tile list that the GEMM launches of (R rows, E experts) read from ws when they are told its list_tile_rows.
int moe_gemm_tile_list(int R, int E, int tile_rows, int ncb_gateup, int ncb_down, int kb, void* ws, size_t ws_bytes, TileList* list) {
  MOE_REQUIRE(ws && list, MOE_ERR_NULL, "gemm tiles: null pointer");
  MOE_REQUIRE(E >= 1 && E <= 1024 && R >= 0, MOE_ERR_BAD_SHAPE, "gemm tiles: need 1 <= E <= 1024, got E=%d R=%d", E, R);
  MOE_REQUIRE(ws_bytes >= moe_gemm_workspace_bytes(R, E, 0), MOE_ERR_WORKSPACE_TOO_SMALL, "gemm tiles: workspace too small");
  *list = tile_list(ws, R, E, tile_rows, ncb_gateup, ncb_down, kb);
  return MOE_OK;
}
