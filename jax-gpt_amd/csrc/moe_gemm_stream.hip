// The grouped GEMMs' kernel for short row tiles: weight streams whose work items are many and short.
//
// The class kernel (moe_gemm.hip) keeps one workgroup on a CU, with all of its LDS as one deep ring.  An item of few K steps
// then spends as long on its start (list entry, row ids, first copies) and its end as on its stream, and nobody on the CU
// streams meanwhile.  Here two workgroups share a CU, each with rings of one or (items of up to 32 rows, moe_stream_depth) two
// stages, so that one streams while the other starts or ends; there is more than one SIMD's worth of waves to hide a step's
// latencies, and the loop is rolled.
// Wave w copies the weight rows that it alone multiplies and takes its fragments to registers as a step begins: the rows'
// place is free at once and is refilled in mid-step, with no barrier, so one stage is nearly always in flight.  The activation
// tile is shared by all waves: one barrier a step, and one stage more than the weights' ring.
//   What bounds it: the HBM (7.0 TB/s of weights at one row an expert, less what the output's writes cost).  Measured against
// the class kernel, gate/up and down: 512 experts of 1024 x 512, 3 rows 92 -> 83 and 52 -> 44 us, 20 rows 101 -> 92 and 60 ->
// 54; 128 of 2048 x 768, 8 rows 66.8 -> 63.9 and 39.4 -> 35.2 (Qwen3-MoE, 33 tokens, all launches 111 -> 104); 32 of
// 7168 x 2048, 2 rows 175 -> 163 for both with list and combine; 128 of 7168 x 2048, whose items are long, within 1 %.
#include "moe_gemm_device.h"

namespace {

constexpr int WAVES = 8, NT = 64 * WAVES;
constexpr int NW = 16 / WAVES;       // weight fragments of 16 rows per wave
constexpr int RG = 32 / WAVES;       // weight row groups of 8 rows that a wave copies: those of its own fragments
// LDS: nst weight tiles, nst + 1 activation tiles with their scales (and a pad: 64 scale slots are copied at a time), the
// item's weight block scales
__host__ __device__ constexpr int x_stage_bytes(int bm) { return bm * BK + bm * 4 + 256; }
__host__ __device__ constexpr int wscale_off(int nst, int bm) { return nst * W_TILE_BYTES + (nst + 1) * x_stage_bytes(bm); }
// the epilogues stage where the rings were
static_assert(kStreamRows * 256 * 2 <= wscale_off(1, kStreamRows) && 32 * (8 * 4 + BK) <= wscale_off(1, 32), "the epilogue stages inside the rings' space");
// every item's rings and weight scales fit where two stages of 32-row tiles do
static_assert(wscale_off(1, kStreamRows) <= wscale_off(2, 32), "rings of the tallest tile");
static_assert(wscale_off(2, 32) + 2 * MAX_KB * 4 <= 80 * 1024, "two workgroups on a CU");

// One item of up to 32 XF rows.  depth: weight stages of an item of up to 32 rows (1 or 2); a taller one has one.
template <int MODE, int XF, bool ONCE>
__device__ __forceinline__ void stream_item(const Item& item, uint8_t* lds, const GemmOperands& op, int depth) {
  constexpr int BM = 32 * XF, NF = 2 * XF;
  constexpr int X_STAGE = x_stage_bytes(BM), S_OFF = BM * BK;
  const int nst = XF == 1 ? depth : 1;
  // copies per wave and step: its weight rows, activation row groups w, w + WAVES, ... (4 XF in all), and one wave for every
  // 64 rows the scales
  constexpr int X_OPS = (4 * XF + WAVES - 1) / WAVES;
  constexpr bool SHORT = 4 * XF < WAVES;          // waves 4 XF .. copy no activations, and the first of them the scales
  constexpr int S_WAVES = (BM + 63) / 64;
  constexpr int OPS = RG + (SHORT ? 0 : X_OPS);   // ... of a wave that has no more than the others
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, fq = lane >> 4;
  const int K = op.K, N = op.N, KB = K / BK, e = item.expert;
  const GemmScales sc = op.sc;

  const int drow = lane >> 3, dchunk = lane & 7;
  const uint8_t* wmat = op.w0 + (size_t)e * N * K;
  const uint8_t* wmat1 = MODE == MODE_GATEUP ? op.w1 + (size_t)e * N * K : wmat;
  unsigned woff[2];
  {
    int grow = MODE == MODE_GATEUP ? item.col_block * 128 + w * (RG * 4) : item.col_block * 256 + w * (RG * 8);
    if (MODE == MODE_DOWN && grow >= N) grow = N - RG * 8;   // (a half-full last column block: re-read valid rows)
    const int piece = dchunk ^ (drow >> 1);
    woff[0] = (unsigned)(grow + drow) * (unsigned)K + piece * 16;
    woff[1] = (unsigned)(grow + drow) * (unsigned)K + (piece ^ 4) * 16;
  }
  const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)lds);
  auto copy_w = [&](int t, int slot) {
#pragma unroll
    for (int i = 0; i < RG; ++i) {
      const uint8_t* base = MODE == MODE_GATEUP ? (i < RG / 2 ? wmat : wmat1) + (size_t)t * BK + (size_t)(i % (RG / 2)) * 8 * K
                                                : wmat + (size_t)t * BK + (size_t)i * 8 * K;
      const unsigned dst = lds0 + slot * W_TILE_BYTES + (MODE == MODE_GATEUP ? (i < RG / 2 ? 0 : 16) + w * (RG / 2) + i % (RG / 2) : w * RG + i) * 1024u;
      if (ONCE) dma16_nt(base, woff[i & 1], dst);
      else dma16(base, woff[i & 1], dst);
    }
  };
  unsigned xoff[X_OPS];
#pragma unroll
  for (int i = 0; i < X_OPS; ++i) {
    const int r = (i * WAVES + w) * 8 + drow;                  // row within the activation tile (past it: never copied)
    const int piece = dchunk ^ ((r >> 1) & 7);
    int g = item.row_start + min(r, item.row_count - 1);
    if (op.row_ids) g = op.row_ids[g];
    xoff[i] = (unsigned)g * (unsigned)K + piece * 16;
  }
  const int slot0 = SHORT ? 0 : min(w * 64, BM > 64 ? BM - 64 : 0);   // first of the 64 scale slots that this wave copies
  unsigned soff;
  {
    const int p = min(slot0 + lane, BM - 1);   // slots past the tile land in the pad
    const int r = 16 * (p % NF) + p / NF;
    int g = item.row_start + min(r, item.row_count - 1);
    if (op.row_ids && !sc.in_listed) g = op.row_ids[g];
    soff = (unsigned)g * (unsigned)sc.in_row * 4u;
  }
  auto copy_x = [&](int t, int slot) {
    const unsigned st = lds0 + nst * W_TILE_BYTES + slot * X_STAGE;
#pragma unroll
    for (int i = 0; i < X_OPS; ++i)
      if ((i + 1) * WAVES <= 4 * XF || i * WAVES + w < 4 * XF) dma16(op.xq + (size_t)t * BK, xoff[i], st + (i * WAVES + w) * 1024u);
    if (SHORT ? w == 4 * XF : w < S_WAVES) {
      dma4((const uint8_t*)(op.sx + (size_t)t * sc.in_kb), soff, st + S_OFF + slot0 * 4u);
    }
  };
  for (int t = 0; t < nst && t < KB; ++t) {
    copy_x(t, t);
    copy_w(t, t);
  }
  // (loads to registers behind the copies: the first step waits for all of these, where the class kernel copies its scales in front of them)
  float* wscale = (float*)(lds + wscale_off(nst, BM));
  for (int i = tid; i < 2 * KB; i += NT) {
    const int h = i >= KB, kk = h ? i - KB : i;
    float v;
    if (MODE == MODE_GATEUP) v = (h ? op.sw1 : op.sw0)[((size_t)e * (N / 128) + item.col_block) * KB + kk];
    else v = op.sw0[((size_t)e * (N / 128) + min(item.col_block * 2 + h, N / 128 - 1)) * KB + kk];
    wscale[i] = v;
  }
  const float* ws0 = wscale + (MODE == MODE_GATEUP ? 0 : w / (WAVES / 2) * KB);
  const float* ws1 = wscale + KB;   // GATEUP only

  const int lane_off0 = fr * BK + ((fq ^ (fr >> 1)) << 4);         // K bytes [16 fq, +16)
  const int lane_off1 = fr * BK + (((fq + 4) ^ (fr >> 1)) << 4);   // K bytes [64 + 16 fq, +16)
  auto read_frag = [&](const uint8_t* base) {
    const v4i lo = *(const v4i*)(base + lane_off0);
    const v4i hi = *(const v4i*)(base + lane_off1);
    return (v8i){lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
  };
  v4f acc[NW][NF];
#pragma unroll
  for (int f = 0; f < NW; ++f)
#pragma unroll
    for (int j = 0; j < NF; ++j) acc[f][j] = (v4f){0.f, 0.f, 0.f, 0.f};
  const bool more_ops = SHORT ? w <= 4 * XF : w < S_WAVES;
  int ws = 0, xs_slot = 0;   // the rings' current slots
  auto step = [&](int kb, auto more) {
    constexpr bool MORE = decltype(more)::value;
    // this wave's copies of stage kb have landed, and its reads of the stage before are done; then everyone's
    // (copies complete in issue order; behind them, with two stages, those of the next step)
    if (XF > 1 || nst == 1 || kb == KB - 1) wait_vm<0>();
    else if (more_ops) wait_vm<OPS + 1>();
    else wait_vm<OPS>();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const int x_next = xs_slot == 0 ? nst : xs_slot - 1;   // the slot of step kb - 1
    if (MORE) copy_x(kb + nst, x_next);
    v8i wf[NW];
#pragma unroll
    for (int f = 0; f < NW; ++f)
      wf[f] = read_frag(lds + ws * W_TILE_BYTES + (MODE == MODE_GATEUP ? (f / (NW / 2) * 128 + w * (NW * 8) + f % (NW / 2) * 16) : (w * (NW * 16) + f * 16)) * BK);
    const float s0 = ws0[kb], s1 = MODE == MODE_GATEUP ? ws1[kb] : s0;
    const uint8_t* xs = lds + nst * W_TILE_BYTES + xs_slot * X_STAGE;
    float sxv[NF];
    if constexpr (NF % 4 != 0) {
#pragma unroll
      for (int j = 0; j < NF; j += 2) {
        const float2 a = *(const float2*)(xs + S_OFF + (fr * NF + j) * 4);
        sxv[j] = a.x, sxv[j + 1] = a.y;
      }
    } else {
#pragma unroll
      for (int j = 0; j < NF; j += 4) {
        const v4f a = *(const v4f*)(xs + S_OFF + (fr * NF + j) * 4);
        sxv[j] = a[0], sxv[j + 1] = a[1], sxv[j + 2] = a[2], sxv[j + 3] = a[3];
      }
    }
    if (MORE) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the weight fragments are in registers: the tile may be overwritten
      copy_w(kb + nst, ws);
    }
    ws = ws + 1 == nst ? 0 : ws + 1;
    xs_slot = xs_slot == nst ? 0 : xs_slot + 1;
#pragma unroll
    for (int j = 0; j < NF; ++j) {
      const v8i xf = read_frag(xs + j * 16 * BK);
      const float c0 = sxv[j] * s0, c1 = sxv[j] * s1;
#pragma unroll
      for (int f = 0; f < NW; ++f) {
        const v4f p = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[f], xf, (v4f){0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
        acc[f][j] += p * ((MODE == MODE_GATEUP && f >= NW / 2) ? c1 : c0);
      }
    }
  };
  int kb = 0;
  for (; kb < KB - nst; ++kb) step(kb, std::true_type{});
  for (; kb < KB; ++kb) step(kb, std::false_type{});
  __syncthreads();   // every wave is done reading before the epilogue reuses LDS
  item_epilogue<MODE, NW, NF, BM, 16, NT>(acc, item, fr, w, lds, N, op.out, op.out_scale, sc);
}

// STREAM: weights come from memory, and those of experts of one row tile are marked as read once (grouped_gemm_kernel).
// rows: of all routed groups.
template <int MODE, bool DENSE, bool STREAM, int MAXXF>
__global__ __launch_bounds__(NT, 4) void stream_gemm_kernel(const GemmOperands routed, TileHeader* hdr, const TileEntry* __restrict__ tiles,
                                                           int rows, const GemmOperands dense, int dense_rows, int dense_tiles,
                                                           int dense_blocks) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const bool is_dense = DENSE && (int)blockIdx.x < dense_blocks;
  const GemmOperands op = is_dense ? dense : routed;
  Item item;
  if (!work_item<MODE, DENSE>(item, lds, op.N, is_dense, hdr, tiles, dense_rows, dense_tiles, dense_blocks)) return;
  auto ncb = [](int N) { return MODE == MODE_GATEUP ? N / 128 : (N + 255) / 256; };
  const int listed = !DENSE || hdr ? hdr->n_tiles : 0;
  const int depth = __builtin_amdgcn_readfirstlane(moe_stream_depth(
      MODE, MAXXF == 1, listed + (DENSE ? dense_tiles : 0), listed * ncb(routed.N) + (DENSE ? dense_tiles * ncb(dense.N) : 0), rows + (DENSE ? dense_rows : 0)));
  const bool once = STREAM && __builtin_amdgcn_readfirstlane(item.tiles) == 1;
#define MOE_CLASS(XF) if (once) stream_item<MODE, XF, true>(item, lds, op, depth); else stream_item<MODE, XF, false>(item, lds, op, depth)
  if constexpr (MAXXF == 1) {
    MOE_CLASS(1);
  } else {
    switch ((__builtin_amdgcn_readfirstlane(item.row_count) + 31) >> 5) {
      case 4: MOE_CLASS(4); break;
      case 3: MOE_CLASS(3); break;
      case 2: MOE_CLASS(2); break;
      default: MOE_CLASS(1); break;
    }
  }
#undef MOE_CLASS
}

template <int MODE, int MAXXF>
int launch(const StreamLaunch& l, hipStream_t s) {
  static std::atomic<unsigned long long> lds_raised[4] = {};
  auto* kernel = l.dense_blocks ? (l.from_memory ? stream_gemm_kernel<MODE, true, true, MAXXF> : stream_gemm_kernel<MODE, true, false, MAXXF>)
                                : (l.from_memory ? stream_gemm_kernel<MODE, false, true, MAXXF> : stream_gemm_kernel<MODE, false, false, MAXXF>);
  const int kb = (l.routed.K > l.dense.K ? l.routed.K : l.dense.K) / BK;
  // (the same for one stage: a third workgroup on the CU makes launches of many items 1 to 4 % slower)
  const int bytes = wscale_off(2, 32) + 2 * kb * (int)sizeof(float);
  if (int rc = moe_raise_lds_limit((const void*)kernel, 80 * 1024, lds_raised[(l.dense_blocks ? 2 : 0) + l.from_memory])) return rc;
  hipLaunchKernelGGL(kernel, dim3(l.grid), dim3(NT), bytes, s, l.routed, l.hdr, l.tiles, l.rows, l.dense, l.dense_rows,
                     l.dense_tiles, l.dense_blocks);
  return moe_check_hip(hipGetLastError(), "gemm launch");
}

}  // namespace

// Where the class kernel is left for this one.  tile_rows: of the tallest tile; items: work items at most (groups that may
// have rows, times column blocks).
//  - Fewer items than 1.5 a CU: a workgroup of its own on each CU and a deep ring are better (8 experts of 7168 x 2048, 1 token,
//    gate/up 48 us; 50 here with two stages, 75 with one).
//  - Gate/up of tiles above 32 rows: its items are longer, and rounds over 2 x 256 workgroups do not come out even (128 experts
//    of 2048 x 768, 60 rows 75.7 us, 79.4 here).  The down GEMM's items are half as long or less: 49.9 -> 45.5.
bool moe_gemm_streams(int mode, int tile_rows, long long items) {
  return items >= kStreamItems && tile_rows <= (mode == MODE_GATEUP ? 32 : kStreamRows);
}
int moe_gemm_stream_launch(int mode, const StreamLaunch& l, hipStream_t s) {
  if (mode == MODE_GATEUP) return launch<MODE_GATEUP, 1>(l, s);
  return l.tile_rows <= 32 ? launch<MODE_DOWN, 1>(l, s) : launch<MODE_DOWN, kStreamRows / 32>(l, s);
}
