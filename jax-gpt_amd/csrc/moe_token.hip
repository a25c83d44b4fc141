// The experts of single tokens: gate/up, then down and combine, without a sort, a work list or y rows.
//
// A token's k experts (and the shared one) are k independent products of one row, so nothing has to be grouped: a workgroup
// takes its expert from the selection itself.  Replaces jax_gpt/models/qwen35/moe.py:58-94 (sort, grouped SwiGLU, scatter
// back), :225-232 and :281 for that batch size.  The grouped GEMMs' arithmetic, instruction for instruction (the same bits):
// one v_mfma_f32_16x16x128_f8f6f4 a scale block, f32 accumulation on the vector ALU, SwiGLU in f32, 1x128 e4m3 quantisation
// of h, bf16 rows, f32 sums in slot order.
//   What bounds it: the stream of the experts' weights, and in small layers each launch's start and its chain of dependent
// loads.  The grouped kernels give one token k * I / 128 work items of 256 weight rows (144 of the DeepSeek-V3 layer, 48 of
// the Qwen3-MoE layer, on 256 CUs) because a quantisation group of h must not cross workgroups.  Here h stays in f32 between
// the two launches and every wave of the second quantises the row that it multiplies -- a few KB from L2 -- so the first
// launch's workgroups can be single waves of 16 columns (1152 and 384).  In the second a workgroup owns tiles of 16 output
// columns of a token, one wave a slot, and adds the slots up itself: no y, no third launch.  Against the grouped route (us a
// call): one token of the DeepSeek-V3 layer 82 -> 68, of Qwen3-MoE 29.3 -> 14.7, of the full layer behind its norm 55.4 -> 42.5, of mini behind
// its norm 18.1 -> 12.5, of tiny 13.7 -> 9.1; five tokens of Qwen3-MoE 44.0 -> 33.0, eight 56.3 -> 46.8; sixteen of mini 23.0 -> 20.6, of tiny
// 14.9 -> 11.1.
//   Rings of two stages, of one or two K steps each (launch_gateup, launch_down); more of them lose or change nothing (of one
// K step, one token of DeepSeek-V3: rings of 2 / 3 / 4 / 6 75.6 / 76.8 / 78.1 / 88.2 in the first launch; in the second 2 / 3 are
// even and 4 / 8 are 7 and 23 % slower).  Workgroups of four waves in the first: 85.8, as 288 of them are uneven on 256 CUs.
//   Where the CUs' LDS holds all workgroups of the first launch they route, and quantise, their token themselves (token_route_gateup_kernel,
// token_front_gateup_kernel): the same work in each, but on otherwise idle CUs, and one launch less.
//   Nothing that a wave has to wait for stands behind the weights' copies, which complete in order with everything else (but the rows of
// further slots of a wave of the second launch, and what a row has beyond 2048 values): codes and scales are copied to LDS in front of them, and the second launch's wave has its whole row of h in registers (2048 values at a time) while the
// selection's index travels, and quantises it while the first weights do.  With loads through registers behind the copies, and h piece by
// piece (us a call): one token of DeepSeek-V3 73.8 -> 70.3, of the full layer 34.6 -> 32.3, of Qwen3-MoE 18.2 -> 17.0, of tiny 12.9 ->
// 11.8, of the mini layer behind its norm 15.3 -> 15.0; 8 tokens of 2 of 8 experts of 1024 x 256 beside one of 4096 30.6 -> 24.2.
#include "moe_token.h"
#include "moe_front_device.h"

namespace {

constexpr int BK = 128;
constexpr int COLS = 16;         // output columns of a wave
constexpr int STAGES = 2;        // of a wave's ring
constexpr int DOWN_TILES = 16;   // most tiles of a workgroup of the second launch
constexpr int kLds = 160 * 1024, kDownLds = kLds - 8192;   // (the second launch has 5.3 KB of static LDS)

template <int N> __device__ __forceinline__ void wait_copies() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// ONCE: weight copies are marked as read once (non-temporal), also those of the shared expert, which every token of the call
// reads: with plain copies of these 2 tokens of the full layer take 55.2 us for 56.6 and of D 2048, 2 of 64 experts of 512 beside
// one of 4096 31.2 for 32.3, but 3 tokens of D 7168, 2 of 24 experts of 512 beside one of 512 41.4 for 39.7 and 16 of D 2048
// 31.6 for 30.7; the other sizes tried are even.
// One wave's products of a row with tiles of FRAGS fragments of 16 weight rows, each fragment of a matrix of its own and the
// tiles `stride` bytes apart: one stream of stages of KS K steps (1 or 2) through a ring, also from one tile to the next.
// LDS: rows of 128 KS bytes, 16-byte chunk c of row r at c ^ ((r >> 1) & 7), as in the grouped kernels, or at c ^ r in rows of 256.
template <int FRAGS, bool ONCE, int KS>
struct WaveRows {
  static constexpr int OPS = 2 * KS, ROW = KS * BK, ROWS = 8 / KS;   // copies of a fragment and stage, bytes and rows of one
  static constexpr int FRAG = 16 * ROW;
  const uint8_t* w[FRAGS];   // the next stage to copy
  unsigned off[OPS];
  unsigned lds;              // the ring's LDS address
  int KB, left, to_copy, copy_kb, slot, KM;
  size_t next_tile;          // from a tile's last stage to the next one's first

  __device__ __forceinline__ void start(const uint8_t* const (&rows)[FRAGS], int K, int tiles, size_t stride, unsigned ring) {
    const int lane = threadIdx.x & 63;
    KB = K / BK, KM = KB / KS, lds = ring, left = to_copy = tiles * KM, copy_kb = 0, slot = 0, next_tile = stride - (size_t)(K - ROW);
#pragma unroll
    for (int f = 0; f < FRAGS; ++f) w[f] = rows[f];
#pragma unroll
    for (int g = 0; g < OPS; ++g) {
      const int r = g * ROWS + lane / (8 * KS), at = lane % (8 * KS);
      off[g] = (unsigned)r * (unsigned)K + (at ^ (KS == 1 ? (r >> 1) & 7 : r)) * 16;
    }
    for (int t = 0; t < STAGES && to_copy; ++t) copy(t);
  }
  __device__ __forceinline__ void copy(int to) {
    const size_t step = ++copy_kb == KM ? next_tile : ROW;
    if (copy_kb == KM) copy_kb = 0;
#pragma unroll
    for (int f = 0; f < FRAGS; ++f) {
#pragma unroll
      for (int g = 0; g < OPS; ++g) {
        const unsigned dst = lds + (unsigned)(to * FRAGS + f) * FRAG + g * 1024u;
        if (ONCE) dma16_nt(w[f], off[g], dst);
        else dma16(w[f], off[g], dst);
      }
      w[f] += step;
    }
    --to_copy;
  }
  // The next tile.  codes: the row's K codes in LDS; scale(kb, f): the product of its scale and the weights' for fragment f
  template <class Scale>
  __device__ __forceinline__ void run(const uint8_t* ring, const uint8_t* codes, v4f (&acc)[FRAGS], const Scale& scale) {
    const int lane = threadIdx.x & 63, fr = lane & 15, fq = lane >> 4;
    for (int km = 0; km < KM; ++km, --left) {
      if (left > 1) wait_copies<OPS * FRAGS>();     // the next stage's copies may be under way
      else wait_copies<0>();
      static_assert(STAGES == 2, "");
      v8i wf[KS][FRAGS];
#pragma unroll
      for (int i = 0; i < KS; ++i)
#pragma unroll
        for (int f = 0; f < FRAGS; ++f) {
          const uint8_t* base = ring + (slot * FRAGS + f) * FRAG + fr * ROW;
          const int x = KS == 1 ? fr >> 1 : fr;
          const v4i lo = *(const v4i*)(base + (((8 * i + fq) ^ x) << 4)), hi = *(const v4i*)(base + (((8 * i + 4 + fq) ^ x) << 4));
          wf[i][f] = (v8i){lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        }
      if (to_copy) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the fragments are in registers: the stage may be overwritten
        copy(slot);
      }
      slot = slot + 1 == STAGES ? 0 : slot + 1;
#pragma unroll
      for (int i = 0; i < KS; ++i) {
        const int kb = km * KS + i;
        // all sixteen columns of the matrix instruction are this row: the lanes of a quarter read one address
        const v4i lo = *(const v4i*)(codes + kb * BK + fq * 16), hi = *(const v4i*)(codes + kb * BK + 64 + fq * 16);
        const v8i xf = (v8i){lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
        for (int f = 0; f < FRAGS; ++f) {
          const v4f p = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[i][f], xf, (v4f){0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
          acc[f] = __builtin_elementwise_fma(p, (v4f)(scale(kb, f)), acc[f]);
        }
      }
    }
  }
};

// LDS of the first launch: ring, the row's codes, its scales and the weights' (copied 64 pieces at a time: whole KB, 256 bytes)
__host__ __device__ constexpr int up_codes(int D) { return (D + 1023) & ~1023; }
__host__ __device__ constexpr int up_scales(int D) { return (D / BK * 4 + 255) & ~255; }
__host__ __device__ constexpr int up_lds(int D, int ks = 1) { return STAGES * 32 * BK * ks + up_codes(D) + 3 * up_scales(D); }
// `n` floats to LDS, 64 at a time
__device__ __forceinline__ void copy_floats(const float* from, int n, unsigned to) {
  for (int i = 0; i < n; i += 64) dma4((const uint8_t*)from, min(i + (int)threadIdx.x % 64, n - 1) * 4u, to + i * 4u);
}

// What a wave of the first launch does once its expert is known.  lds: ring, codes, [2] weights' scales (up_lds); the row's scales at sx
template <bool ONCE, int KS>
struct GateUpTile {
  const TokenArgs& a;
  int t, slot, col;
  bool shared;
  uint8_t* lds;
  WaveRows<2, ONCE, KS> rows;
  float *sx, *sw;   // sw: [2][up_scales / 4]

  // Workgroup b of a token's: its slot and columns
  __device__ __forceinline__ GateUpTile(const TokenArgs& args, int b, int token, uint8_t* base, int codes_bytes) : a(args), t(token), lds(base) {
    const int per = a.I / COLS;
    shared = b >= a.k * per;
    slot = shared ? a.k : b / per, col = (b - slot * per) * COLS;
    sx = (float*)(base + STAGES * 32 * BK * KS + codes_bytes), sw = sx + up_scales(a.D) / 4;
  }
  __device__ __forceinline__ uint8_t* codes() const { return lds + STAGES * 32 * BK * KS; }
  static __device__ __forceinline__ unsigned address(const void* p) { return __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)p); }
  __device__ __forceinline__ void start(int e) {
    const TokenExperts& x = shared ? a.shared : a.routed;
    const int N = shared ? a.SI : a.I, KB = a.D / BK;
    const size_t block = ((size_t)e * (N / BK) + col / BK) * KB;
    copy_floats(x.s_gate + block, KB, address(sw));
    copy_floats(x.s_up + block, KB, address(sw) + up_scales(a.D));
    const size_t row = ((size_t)e * N + col) * a.D;
    rows.start({x.w_gate + row, x.w_up + row}, a.D, 1, 0, address(lds));
  }
  __device__ __forceinline__ void finish() {
    const int lane = threadIdx.x & 63, per_scale = up_scales(a.D) / 4;
    v4f acc[2] = {};
    const float *rs = sx, *ws = sw;
    rows.run(lds, codes(), acc, [&](int kb, int f) { return rs[kb] * ws[f * per_scale + kb]; });
    v4f h;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float g = acc[0][r], u = acc[1][r];
      h[r] = g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)) * u;
    }
    if ((lane & 15) == 0) *(v4f*)(a.h + ((size_t)t * (a.k + 1) + slot) * a.h_stride + col + (lane >> 4) * 4) = h;
  }
};

template <bool ONCE, int KS>
__global__ __launch_bounds__(64) void token_gateup_kernel(const TokenArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int lane = threadIdx.x, t = blockIdx.y;
  GateUpTile<ONCE, KS> tile(a, blockIdx.x, t, lds, up_codes(a.D));
  const int chosen = tile.shared ? 0 : a.idx[(size_t)t * a.k + tile.slot];
  // everything is copied by the wave itself, in the order of its use: what does not depend on the expert while its index travels
  const unsigned codes_at = tile.address(tile.codes());
  for (int i = 0; i < a.D; i += 1024) dma16(a.xq + (size_t)t * a.D, min(i + lane * 16, a.D - 16), codes_at + i);
  copy_floats(a.sx + (size_t)t * (a.D / BK), a.D / BK, tile.address(tile.sx));
  const int e = __builtin_amdgcn_readfirstlane(chosen);
  if (!tile.shared && (unsigned)e >= (unsigned)a.E) {   // (an index out of range: the second launch leaves its row out)
    wait_copies<0>();   // (none may land in LDS that is another workgroup's)
    return;
  }
  tile.start(e);
  tile.finish();
}

// A piece of eight values of a token's row to its codes and scale in LDS; 16 lanes a group
__device__ __forceinline__ void quant_piece(const moe_bf16x8& in, int p, uint8_t* codes, float* sx) {
  float scale_inv;
  ((uint2*)codes)[p] = front_codes(in, scale_inv);
  if ((p & 15) == 0) sx[p >> 4] = scale_inv;
}
// LDS writes of all waves are there; the copies stay under way
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// The same with the token's routing and quantisation in front, from ready logits (or a given selection): the first wave selects its token's experts itself
// and streams their weights, the others quantise the token meanwhile (rows above 4096: two of them).  What it waits for is the
// selection's chain of dependent steps, as the launch before did, without that launch's end and this one's start.  One token of
// DeepSeek-V3, launch by launch 71.0 us a call; this way with the selecting wave quantising behind its first copies 71.0 (110
// instructions for 512 values), with one wave for that 70.2, with two 68.5, three 68.8.
constexpr int SELECTED = -1;   // (a KIND: nothing to route)
template <int KIND, int VPL, bool ONCE, int KS>
__global__ __launch_bounds__(192) void token_route_gateup_kernel(const TokenArgs a, const RouteArgs r, const bf16_t* x) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int lane = threadIdx.x & 63, t = blockIdx.y, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  GateUpTile<ONCE, KS> tile(a, blockIdx.x, t, lds, up_codes(a.D));
  if (w > 0) {
    const moe_bf16x8* row = (const moe_bf16x8*)(x + (size_t)t * a.D);
    for (int p = threadIdx.x - 64; p < a.D / 8; p += blockDim.x - 64) quant_piece(row[p], p, tile.codes(), tile.sx);
    lds_barrier();
    return;
  }
  Chosen chosen{};
  int e = 0;
  if (KIND == SELECTED) {
    if (!tile.shared) e = __builtin_amdgcn_readfirstlane(a.idx[(size_t)t * a.k + tile.slot]);
    if (!tile.shared && (unsigned)e >= (unsigned)a.E) {   // (out of range: the second launch leaves its row out)
      lds_barrier();
      return;
    }
  } else if (!tile.shared) {
    const float* row = r.src.logits + (size_t)t * a.E;
    chosen = KIND == ROUTE_SOFTMAX ? route_softmax_token<VPL>(r, row, t, false) : route_grouped_token<VPL>(r, row, t, false);
    e = __builtin_amdgcn_readlane(chosen.expert, tile.slot);
  }
  tile.start(e);
  lds_barrier();
  tile.finish();
  if (KIND != SELECTED && blockIdx.x == 0 && lane < a.k) r.idx[(size_t)t * a.k + lane] = chosen.expert, r.w[(size_t)t * a.k + lane] = chosen.weight;
}

// The same behind a small router (front_kernel, whose sums, blocks and instructions these are): the workgroup's eight waves norm the
// token and multiply a K block of the router each, and the first goes on alone with the selection and its experts' weights.  Bound by
// its start and the chain behind it: mini layer behind its norm, one token, 14.8 us a call in three launches, 12.8 in two.
constexpr int FRONT_WAVES = 8, FRONT_COLUMNS = 65;
__host__ __device__ constexpr int front_up_lds(int D, int N, int ks) { return up_lds(D, ks) + D * 2 + (N * (D / 128 + 1) + 3) / 4 * 16; }
template <int KIND, bool NORM, int KS>
__global__ __launch_bounds__(64 * FRONT_WAVES) void token_front_gateup_kernel(const TokenArgs a, const RouteArgs r, const FrontArgs f) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];   // [the tile's][the row's pieces][the K blocks' products][logits]
  constexpr int GROUPS = (FRONT_COLUMNS + 15) / 16;
  __shared__ float wave_sum[2];
  const int tid = threadIdx.x, lane = tid & 63, t = blockIdx.y, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, fq = lane >> 4, N = r.src.N, E = a.E, D = a.D, KB = D / BK, P = D / 8;
  GateUpTile<false, KS> tile(a, blockIdx.x, t, lds, up_codes(D));
  v4i* pieces = (v4i*)(lds + up_lds(D, KS));
  float *products = (float*)(pieces + P), *logits = products + KB * N;
  // the row's pieces: the last wave has the first 64, the one before it the rest
  const int unit = FRONT_WAVES - 1 - w, p = unit * 64 + lane;
  const bool has = unit < 2 && p < P;
  moe_bf16x8 in = {};
  v4f wt[2] = {};
  if (has) {
    in = load_bf16x8(f.x, f.x_f32, (size_t)t * P + p);
    if (NORM) wt[0] = ((const v4f*)f.norm)[2 * p], wt[1] = ((const v4f*)f.norm)[2 * p + 1];
  }
  v4i b[GROUPS][4];
  if (w < KB) front_weights(b, (const bf16_t*)f.w_router, (const bf16_t*)f.w_shared_gate, E, N, D, w);
  if (NORM) {
    if (unit < 2) {
      const float ss = wave_sum_f32(front_squares(in));
      if (lane == 0) wave_sum[unit] = ss;
    }
    lds_barrier();
    front_norm(in, P > 64 ? __fadd_rn(wave_sum[0], wave_sum[1]) : wave_sum[0], D, f.eps, wt);
  }
  if (has) pieces[p] = __builtin_bit_cast(v4i, in);
  lds_barrier();
  if (w < KB) {
    v4i av[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) av[s] = pieces[w * 16 + 4 * s + fq];   // (all sixteen rows of the matrix instruction are this one)
#pragma unroll
    for (int g = 0; g < GROUPS; ++g) {
      if (16 * g >= N) break;
      const v4f acc = front_products(av, b[g]);
      if (fq == 0 && 16 * g + fr < N) products[w * N + 16 * g + fr] = acc[0];
    }
  }
  lds_barrier();
  if (has) quant_piece(in, p, tile.codes(), tile.sx);
  if (tid < 128)   // (N <= 65)
    if (tid < N) logits[tid] = front_logit(products + tid, KB, N);
  lds_barrier();
  if (w > 0) return;
  Chosen chosen{};
  int e = 0;
  if (!tile.shared) {
    chosen = KIND == ROUTE_SOFTMAX ? route_softmax_token<1>(r, logits, t, false) : route_grouped_token<1>(r, logits, t, false);
    e = __builtin_amdgcn_readlane(chosen.expert, tile.slot);
  }
  tile.start(e);
  tile.finish();
  if (blockIdx.x == 0) {   // (a routed tile: it has the selection)
    if (lane < a.k) r.idx[(size_t)t * a.k + lane] = chosen.expert, r.w[(size_t)t * a.k + lane] = chosen.weight;
    if (r.src.out_logits && lane < E) r.src.out_logits[(size_t)t * E + lane] = logits[lane];
    if (lane == 0 && r.src.shared_gate && N > E) r.src.shared_gate[t] = front_gate(logits[E]);
  }
}

// LDS of a wave of the second launch: ring, codes and scales of its row, the weights' scales of its tiles
__host__ __device__ constexpr int down_wave_lds(int I, int tiles, int ks = 1) {
  return STAGES * 16 * BK * ks + I + (I / BK * 4 + 15) / 16 * 16 + ((tiles * (I / BK) + 63) / 64 * 256);
}

// with the lane that CTRL pairs this one with, in one instruction (0 from outside)
template <int CTRL> __device__ __forceinline__ unsigned max_dpp(unsigned v) {
  return max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true));
}
constexpr int H_PIECES = 8;   // of four values a lane: 2048 of a row

// A workgroup: `tiles` neighbouring tiles of 16 output columns of a token; a wave: a slot's row (several, if there are more
// slots than waves; then tiles is 1).
template <bool ONCE, int KS>
__global__ __launch_bounds__(1024) void token_down_kernel(const TokenArgs a, const int tiles) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  __shared__ float y[2][MOE_TOKEN_SLOTS][COLS];
  __shared__ float weight[MOE_TOKEN_SLOTS];
  __shared__ float residual[DOWN_TILES * COLS];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
  const int t = blockIdx.y, first = blockIdx.x * tiles, count = min(tiles, a.D / COLS - first), slots = a.k + (a.SI > 0);
  uint8_t* ring = lds + w * down_wave_lds(a.h_stride, tiles, KS);
  uint8_t* codes = ring + STAGES * 16 * BK * KS;
  float* sx = (float*)(codes + a.h_stride);
  const int sw_at = STAGES * 16 * BK * KS + a.h_stride + (a.h_stride / BK * 4 + 15) / 16 * 16;
  const float* sw = (const float*)(ring + sw_at);   // [tile][kb]
  const unsigned ring_at = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)ring);
  // What the sums need, and what a wave needs first: all under way before anything is waited for (copies come behind them).
  float wv = 0.f;
  unsigned rv[DOWN_TILES * COLS / 64];   // (bits, converted below: a conversion would wait here)
  if (w == waves - 1) {
    if (lane < a.k) wv = a.w[(size_t)t * a.k + lane];
    else if (a.shared_gate && lane == a.k) wv = a.shared_gate[t];
    const size_t at = (size_t)t * a.D + first * COLS;
    if (a.residual)
#pragma unroll
      for (int i = 0; i < DOWN_TILES * COLS / 64; ++i)
        if (i * 64 + lane < count * COLS)
          rv[i] = a.io_f32 ? ((const unsigned*)a.residual)[at + i * 64 + lane] : ((const bf16_t*)a.residual)[at + i * 64 + lane];
  }
  // the slot's row of h, some of it in registers: the loads of the first slot are under way before its expert is known
  v4f hv[H_PIECES];
  auto load_h = [&](int slot, int from) {
    const int n = (slot == a.k ? a.SI : a.I) / 4;
    const v4f* h = (const v4f*)(a.h + ((size_t)t * (a.k + 1) + slot) * a.h_stride);
#pragma unroll
    for (int i = 0; i < H_PIECES; ++i)
      if (from + 64 * i < n) hv[i] = h[min(from + 64 * i + lane, n - 1)];
  };
  WaveRows<1, ONCE, KS> rows;
  int e = w < a.k ? a.idx[(size_t)t * a.k + w] : 0;   // (of the wave's only slot, where there are several tiles)
  if (w < slots) load_h(w, 0);
  e = __builtin_amdgcn_readfirstlane(e);
#pragma unroll
  for (int i = 0; i < H_PIECES; ++i) asm volatile("" : "+v"(hv[i]));   // (waited for before copies are under way, and not behind them)
  if (w == waves - 1) {
    if (lane < slots) weight[lane] = wv;
    if (a.residual)
#pragma unroll
      for (int i = 0; i < DOWN_TILES * COLS / 64; ++i)
        if (i * 64 + lane < count * COLS) residual[i * 64 + lane] = bf16_to_f32(a.io_f32 ? f32_to_bf16(__uint_as_float(rv[i])) : (bf16_t)rv[i]);
  }
  for (int j = 0; j < count; ++j) {
    for (int slot = w; slot < slots; slot += waves) {
      const bool shared = slot == a.k;
      const int K = shared ? a.SI : a.I, KB = K / BK;
      if (slot != w) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (the last slot's reads are done before copies land where they read)
        e = __builtin_amdgcn_readfirstlane(shared ? 0 : a.idx[(size_t)t * a.k + slot]);
      }
      v4f acc[1] = {};
      if (shared || (unsigned)e < (unsigned)a.E) {
        if (j == 0) {
          const TokenExperts& x = shared ? a.shared : a.routed;
          for (int i = 0; i < count * KB; i += 64) {
            const int at = min(i + lane, count * KB - 1), tile = at / KB;
            dma4((const uint8_t*)(x.s_down + (size_t)e * (a.D / BK) * KB), (unsigned)((first + tile) * COLS / BK * KB + at - tile * KB) * 4u,
                 ring_at + sw_at + i * 4u);
          }
          rows.start({x.w_down + ((size_t)e * a.D + first * COLS) * K}, K, count, (size_t)COLS * K, ring_at);
          // the row's quantisation groups, 32 lanes each (the maximum by lane permutations: where a wave has two slots the launch waits
          // for its instructions, and with five shuffles 16 tokens of 32 of 256 experts of 1024 x 128 took 25.9 us for 24.0)
          for (int from = 0; from < K / 4; from += 64 * H_PIECES) {
            if (from || slot != w) load_h(slot, from);
#pragma unroll
            for (int p = 0; p < H_PIECES; ++p) {
              const int i = from + 64 * p + lane;
              if (from + 64 * p >= K / 4) break;
              const v4f v = hv[p];   // (lanes past the row's end: half a wave, whose group is its own)
              float amax = 0.f;
#pragma unroll
              for (int r = 0; r < 4; ++r) amax = fmaxf(amax, fabsf(v[r]));
              unsigned m = __float_as_uint(amax);   // (not negative: ordered as integers)
              m = max_dpp<DPP_XOR1>(m);
              m = max_dpp<DPP_XOR2>(m);
              m = max_dpp<DPP_MIRROR8>(m);
              m = max_dpp<DPP_MIRROR16>(m);
              const auto pair = __builtin_amdgcn_permlane16_swap(m, m, false, false);   // (even rows of 16 lanes twice, and odd ones)
              m = max(pair[0], pair[1]);
              float scale, scale_inv;
              fp8_scales(__uint_as_float(m), scale, scale_inv);
              int q = 0;
              q = __builtin_amdgcn_cvt_pk_fp8_f32(__builtin_amdgcn_fmed3f(v[0] * scale, -MOE_FP8_MAX, MOE_FP8_MAX),
                                                  __builtin_amdgcn_fmed3f(v[1] * scale, -MOE_FP8_MAX, MOE_FP8_MAX), q, false);
              q = __builtin_amdgcn_cvt_pk_fp8_f32(__builtin_amdgcn_fmed3f(v[2] * scale, -MOE_FP8_MAX, MOE_FP8_MAX),
                                                  __builtin_amdgcn_fmed3f(v[3] * scale, -MOE_FP8_MAX, MOE_FP8_MAX), q, true);
              if (i < K / 4) {
                ((int*)codes)[i] = q;
                if ((i & 31) == 0) sx[i >> 5] = scale_inv;
              }
            }
          }
        }
        rows.run(ring, codes, acc, [&](int kb, int) { return sx[kb] * sw[j * KB + kb]; });
      }
      if ((lane & 15) == 0) {   // the row in bf16
        const unsigned lo = pack2_bf16(acc[0][0], acc[0][1]), hi = pack2_bf16(acc[0][2], acc[0][3]);
        float* dst = y[j & 1][slot] + 4 * (lane >> 4);
        dst[0] = __uint_as_float(lo << 16), dst[1] = __uint_as_float(lo & 0xffff0000u);
        dst[2] = __uint_as_float(hi << 16), dst[3] = __uint_as_float(hi & 0xffff0000u);
      }
    }
    // this tile's rows are there (and those of the one before have been read: the sums below precede the next barrier);
    // copies stay under way
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (tid < COLS) {
#pragma clang fp contract(off)
      float s = 0.f;
      for (int i = 0; i < a.k; ++i) s = s + y[j & 1][i][tid] * weight[i];
      if (a.SI > 0) s = s + (a.shared_gate ? y[j & 1][a.k][tid] * weight[a.k] : y[j & 1][a.k][tid]);
      if (a.residual) s = s + residual[j * COLS + tid];
      const size_t at = (size_t)t * a.D + (first + j) * COLS + tid;
      const bf16_t o = f32_to_bf16(s);
      if (a.io_f32) ((float*)a.out)[at] = bf16_to_f32(o);
      else ((bf16_t*)a.out)[at] = o;
    }
  }
}

int launch_gateup(const TokenArgs& a, bool from_memory, hipStream_t s) {
  static std::atomic<unsigned long long> raised[4] = {};
  const bool pairs = moe_token_stages(a.M, a.D, a.k, a.I, a.SI, from_memory).gateup == 2;
  auto* kernel = pairs ? (from_memory ? token_gateup_kernel<true, 2> : token_gateup_kernel<false, 2>)
                       : (from_memory ? token_gateup_kernel<true, 1> : token_gateup_kernel<false, 1>);
  if (int rc = moe_raise_lds_limit((const void*)kernel, kLds, raised[2 * pairs + from_memory])) return rc;
  hipLaunchKernelGGL(kernel, dim3((a.k * a.I + a.SI) / COLS, a.M), dim3(64), up_lds(a.D, 1 + pairs), s, a);
  return moe_check_hip(hipGetLastError(), "token gate/up launch");
}

template <int KIND, bool ONCE, int KS>
auto route_gateup_kernel(int E) {
  if constexpr (KIND == SELECTED) return token_route_gateup_kernel<KIND, 1, ONCE, KS>;
  else return E <= 128 ? token_route_gateup_kernel<KIND, 2, ONCE, KS> : token_route_gateup_kernel<KIND, 4, ONCE, KS>;
}
template <int KIND>
auto route_gateup_kernel(int E, bool from_memory, bool pairs) {
  return pairs ? (from_memory ? route_gateup_kernel<KIND, true, 2>(E) : route_gateup_kernel<KIND, false, 2>(E))
               : (from_memory ? route_gateup_kernel<KIND, true, 1>(E) : route_gateup_kernel<KIND, false, 1>(E));
}
template <int KIND>
auto front_gateup_kernel(bool norm, bool pairs) {
  return pairs ? (norm ? token_front_gateup_kernel<KIND, true, 2> : token_front_gateup_kernel<KIND, false, 2>)
               : (norm ? token_front_gateup_kernel<KIND, true, 1> : token_front_gateup_kernel<KIND, false, 1>);
}
int launch_route_gateup(const TokenArgs& a, const TokenRoute& route, bool from_memory, hipStream_t s) {
  static std::atomic<unsigned long long> raised[20] = {};
  const int pairs = moe_token_stages(a.M, a.D, a.k, a.I, a.SI, from_memory).gateup == 2;
  const bool softmax = route.routing == MOE_ROUTING_SOFTMAX;
  const dim3 grid((a.k * a.I + a.SI) / COLS, a.M);
  if (route.front) {   // (64 KB of LDS hold these)
    auto* kernel = softmax ? front_gateup_kernel<ROUTE_SOFTMAX>(route.front->norm, pairs) : front_gateup_kernel<ROUTE_GROUPED>(route.front->norm, pairs);
    hipLaunchKernelGGL(kernel, grid, dim3(64 * FRONT_WAVES), front_up_lds(a.D, route.args.src.N, 1 + pairs), s, a, route.args, *route.front);
    return moe_check_hip(hipGetLastError(), "token router and gate/up launch");
  }
  auto* kernel = route.selected ? route_gateup_kernel<SELECTED>(a.E, from_memory, pairs)
                 : softmax      ? route_gateup_kernel<ROUTE_SOFTMAX>(a.E, from_memory, pairs)
                                : route_gateup_kernel<ROUTE_GROUPED>(a.E, from_memory, pairs);
  const int which = route.selected ? 4 : (a.E > 128) * 2 + softmax;
  if (int rc = moe_raise_lds_limit((const void*)kernel, kLds, raised[which * 4 + 2 * pairs + from_memory])) return rc;
  const int quantisers = a.D > 4096 ? 2 : 1;
  hipLaunchKernelGGL(kernel, grid, dim3(64 * (1 + quantisers)), up_lds(a.D, 1 + pairs), s, a, route.args, (const bf16_t*)route.x);
  return moe_check_hip(hipGetLastError(), "token route and gate/up launch");
}

int down_tiles(int D, int M) {
  const int cols = D / COLS;
  int tiles = 1;
  while (tiles < DOWN_TILES && (cols + tiles - 1) / tiles * M > 256) ++tiles;
  return tiles;
}
int launch_down(const TokenArgs& a, bool from_memory, hipStream_t s) {
  static std::atomic<unsigned long long> raised[4] = {};
  const TokenDownPlan p = moe_token_down_plan(a.M, a.D, a.k, a.I, a.SI);
  const bool pairs = moe_token_stages(a.M, a.D, a.k, a.I, a.SI, from_memory).down == 2;
  auto* kernel = pairs ? (from_memory ? token_down_kernel<true, 2> : token_down_kernel<false, 2>)
                       : (from_memory ? token_down_kernel<true, 1> : token_down_kernel<false, 1>);
  if (int rc = moe_raise_lds_limit((const void*)kernel, kDownLds, raised[2 * pairs + from_memory])) return rc;
  hipLaunchKernelGGL(kernel, dim3((a.D / COLS + p.tiles - 1) / p.tiles, a.M), dim3(64 * p.waves),
                     p.waves * down_wave_lds(a.h_stride, p.tiles, 1 + pairs), s, a, p.tiles);
  return moe_check_hip(hipGetLastError(), "token down launch");
}

}  // namespace

// Up to a workgroup per CU, each with as many tiles as that takes: a row is quantised once, the copies run on from tile to
// tile, and no CU has a second workgroup of about 80 KB of LDS to begin (full layer, 2 tokens, workgroups of 2 tiles against
// 512 of one: 70.1 / 74.3 us; mini, 8: 31.3 / 32.9; one workgroup more than there are CUs -- 6 tokens of Qwen3-MoE in 258 --
// 46.3 against 43.4 in 192).
TokenDownPlan moe_token_down_plan(int M, int D, int k, int I, int SI) {
  const int slots = k + (SI > 0), widest = I > SI ? I : SI;
  int tiles = down_tiles(D, M);
  if (slots > 16 || slots * down_wave_lds(widest, tiles) > kDownLds) tiles = 1;   // (a wave of several slots)
  const int wave_lds = down_wave_lds(widest, tiles), fit = kDownLds / wave_lds, most = fit < 16 ? fit : 16;
  return {tiles, slots < most ? slots : most, wave_lds};
}

// Every token reads its experts itself, where the grouped kernels read an expert once for all its rows, and a wave of the second
// launch walks its tiles' K steps one after the other.  What the launches left out and the finer split gain (3 to 15 us) covers (us a call,
// grouped / this way)
//  - up to some 320 MB of weights, which 16-row streams read at about 6 TB/s against 6.9 (Qwen3-MoE, 8 tokens = 302 MB 56.3 /
//    46.8, 10 = 377 MB 66.4 / 64.2, 12 = 453 MB 71.5 / 73.5; full layer behind its norm, 2 tokens = 277 MB 72.0 / 65.4, 3 = 415 MB 82.3 /
//    88.0).  The line is from before the launch in front of the experts fell away and is on the careful side (9 tokens of
//    Qwen3-MoE 61.0 / 54.8; DeepSeek-V3, 2 tokens = 793 MB 154 / 125);
//  - of these, megabytes that are read again, and eight times the K steps that the second launch's longest chain has beyond one
//    tile's, up to 300 (of layers that the memory-side cache holds).  A shared expert eight times as
//    wide, D 1024, 2 of 32 experts of 512: 4 tokens (no further steps) 24.8 / 15.1, 8 (32) 26.6 / 20.8, 12 (64) 27.2 / 29.3, 16 (96)
//    28.4 / 34.6.  D 4096, 2 of 4 experts of 1024: 4 tokens (24) 25.7 / 19.0, 8 (56, 144 MB again) 26.0 / 24.9, 12 26.2 / 33.5.
//    8 of 8 experts, D 1024 x 1024: 8 tokens (8, 168 MB) 17.6 / 17.2, 12 (24, 264 MB) 17.8 / 25.5; 8 of 8, 16 and 32 experts of
//    2048 x 768, 8 tokens (18 and 252, 216 and 144 MB) 20.8 / 22.5, 22.8 / 24.8, 32.0 / 34.8.  In 170 drawn layers and batches of 2 to 16
//    tokens the choice by this line is 0.9 % slower than the better route on average (by the first line alone 2.4 %), 41 % at worst: small
//    layers whose down projection is one launch with the combine (moe_small.hip) lose where an expert has many tokens (13 tokens of 8 of 8
//    experts of 512 x 1408 17.1 / 24.2).
// One token reads nothing twice and gains at any size (396 MB of DeepSeek-V3: 82 -> 68).  Above 16 tokens nothing is taken: 24 were even
// with the grouped route when that had three launches more.
bool moe_token_takes(int M, int D, int E, int k, int I, int SI) {
  const int widest = I > SI ? I : SI;
  if (M < 1 || M > MOE_TOKEN_ROWS || k < 1 || k >= MOE_TOKEN_SLOTS || up_lds(D) > kLds || down_wave_lds(widest, 1) > kDownLds) return false;
  if (M == 1) return true;
  const long long touched = (long long)M * k < E ? (long long)M * k : E;
  const long long bytes = 3ll * M * ((long long)k * I + SI) * D, once = 3ll * (touched * I + SI) * D;
  const long long steps = (long long)(down_tiles(D, M) - 1) * (widest / BK);
  return bytes <= (320ll << 20) && 8 * steps + ((bytes - once) >> 20) <= 300;
}

// Two K steps a stage, 256 bytes of a row (us, one / two).  In the first launch
//  - from memory while a CU has up to four workgroups: one token of Qwen3-MoE 19.8 / 17.9 for the call, two 21.8 / 21.2; with more of
//    them their rows get in each other's way: one of DeepSeek-V3 (1152 workgroups) 74.7 / 75.5, 6 of Qwen3-MoE 42.8 / 44.7;
//  - from the caches while the CUs hold all workgroups at once, eight or nine of 17 to 18 KB of LDS (the launch: 32 experts of
//    2048 x 768, k = 8, 1 token 11.0 / 8.2, 4 of it (1536 workgroups) 15.2 / 14.5, 6 (2304) 18.2 / 20.2, 8 21.3 / 24.0; 16 of 1024 x 2048,
//    k = 4, 4 tokens (2048) 11.8 / 11.1, 8 15.1 / 15.9; 8 of 1024 x 1024, k = 8, 8 tokens 9.9 / 11.4); rows of less than 1024 while
//    a CU has up to four (8 of 512 x 1024, k = 2, 5 tokens (640) 5.0 / 4.8, 16 (2048) 5.5 / 5.8; 16 of 512 x 512, k = 16, 1 token 4.9 /
//    4.8, 4 (2048) 5.4 / 5.7, 8 (4096) 6.8 / 8.6).
// In the second one from the caches, or where a wave walks up to 24 K steps: 16 tokens of tiny 16.5 / 15.5 for the call, of the mini layer
// 21.5 / 20.7, 6 of Qwen3-MoE 43.7 / 42.8, 8 50.8 / 50.5, 2 of the full layer 61.5 / 61.1; DeepSeek-V3 (32 steps) 74.5 / 74.7.  (The launch
// of these layers, 1 to 16 tokens: -23 to +2 %.)
TokenStages moe_token_stages(int M, int D, int k, int I, int SI, bool from_memory) {
  const long long workgroups = (long long)M * ((k * I + SI) / COLS);
  const int up = up_lds(D, 2);
  const bool gateup = D % (2 * BK) == 0 && up <= kLds && workgroups <= (from_memory || D < 1024 ? 1024 : 256 * (kLds / up));
  const TokenDownPlan p = moe_token_down_plan(M, D, k, I, SI);
  const int widest = I > SI ? I : SI;
  const bool down = I % (2 * BK) == 0 && SI % (2 * BK) == 0 && p.waves * down_wave_lds(widest, p.tiles, 2) <= kDownLds &&
                    (!from_memory || p.tiles * (widest / BK) <= 24);
  return {1 + gateup, 1 + down};
}

// Ready logits: while the CUs' LDS holds all workgroups, which then route side by side: the launch that falls away took 3.6 to
// 5.7 us and its end and the next one's start between them (us a call, launch by launch / this way): tiny, 1 token 11.3 / 8.9, 16 14.0 /
// 11.6; Qwen3-MoE, 1 16.8 / 14.4, 4 31.4 / 28.7, 8 (3072 workgroups) 50.6 / 48.0; DeepSeek-V3, 1 71.0 / 68.5.  Nothing was measured above
// 256 experts.  A given selection (the launch that falls away is the quantiser's): moe_routing and expert_forward_single of tiny, 1 to 16
// tokens 20.0 / 17.8, of Qwen3-MoE, 1 24.0 / 22.6, 4 37.4 / 36.0, 8 56.7 / 54.8.
//   The selection is a chain of k steps, and of a step for each group where groups lie across lanes, and all workgroups of a CU repeat it:
// up to 48 K steps of them in all, a step of the grouped routing being one and a half; 64 K and, of more than 128 experts, 128 K
// where rows of 1024 and more stream meanwhile.  This way against launch by launch, hidden sizes of 128 to 768: softmax, 32 of 64 or 256 experts,
// 1536 workgroups (48 K) 0.91 to 1.00, 2048 0.93 to 1.05, 3072 0.99 to 1.10, 4096 0.97 to 1.17; 16 of them, 2048 (32 K) 0.87 to 0.92; 8 of 256,
// 4096 (32 K) 0.88 to 0.96.  Grouped, 8 groups: 32, 1024 (48 K) 0.92 to 1.01, 1536 0.96 to 1.07, 4096 1.06 to 1.28; 16, 2048 (48 K)
// 0.90 to 0.97; 8, 4096 (48 K) 0.92 to 1.02.  240 experts in 48 groups of five, k = 8: 512 (42 K) 0.94, 1024 (84 K) 0.94, 2048 1.01 to 1.10,
// 4096 1.15 to 1.57.  D 1024: softmax, 32 of 256 experts, 4096 (128 K) 0.95, of 64, 2048 (64 K) 0.95, 4096 1.04; grouped, 32 of 256, 2560
// (120 K) 0.97, 4096 0.99 to 1.00, 32 of 64, 1024 (48 K) 1.00, 2560 1.08; 16 of 256, 4096 (96 K) 0.95.
int moe_token_chain(int routing, int E, int k, int n_group, int topk_group) {
  if (routing != MOE_ROUTING_SIGMOID_GROUPED) return k;
  const int lane_keys = E <= 128 ? 2 : 4, per = n_group > 0 ? E / n_group : 0, lanes = per / lane_keys;
  const bool across = topk_group < n_group && !(lanes * lane_keys == per && (lanes == 1 || lanes == 2 || lanes == 4 || lanes == 8 || lanes == 16));
  return (k + (across ? n_group : 0)) * 3 / 2;
}
bool moe_token_routes(int M, int D, int E, int k, int I, int SI, bool selected, int chain) {
  const int lds = up_lds(D);
  const long long workgroups = (long long)M * ((k * I + SI) / COLS);
  const long long most = D < 1024 ? 48 : E > 128 ? 128 : 64;
  return (selected || (E <= 256 && workgroups * chain <= most * 1024)) && lds <= kLds && workgroups <= 256 * (kLds / lds);
}
// Behind a small router every workgroup of eight waves repeats the router's matmul.  Mini layer, 96 workgroups a token, launch by
// launch / this way: 1 token 14.0 / 11.6, 4 14.6 / 13.9, 5 15.2 / 14.6, 8 (768 workgroups) 15.4 / 17.9; behind its norm 1 14.8 / 12.8,
// 2 15.1 / 12.9, 3 15.1 / 14.4, 4 15.2 / 15.3, 6 16.3 / 19.8.
//   One workgroup a CU gains with any router (10 to 30 %).  Where some CUs have two, the CU reads the router's weights twice, and the
// line lies at their number (columns x D; this way against launch by launch): 320 to 512 workgroups without a norm, 33 K 0.93 to
// 0.98, 42 K 0.99 to 1.01, 50 K 1.01 to 1.05, 66 K 1.06 to 1.09; behind a norm, 288 to 320, 25 K 0.92 to 0.99, 31 to 34 K 0.96 to 1.01, 44 K
// 1.01 to 1.06, 66 K 1.08 to 1.12.  How many experts are chosen, and of which groups, changes little here.
bool moe_token_fronts(int M, int k, int I, int SI, bool norm, bool from_memory, int router) {
  const long long workgroups = (long long)M * ((k * I + SI) / COLS);
  return !from_memory && (workgroups <= 256 || (workgroups <= (norm ? 320 : 512) && router <= (norm ? 34 : 42) * 1024));
}

int moe_token_experts(const TokenArgs& a, bool from_memory, const TokenRoute* route, moe_stream_t stream) {
  hipStream_t s = (hipStream_t)stream;
  if (int rc = route ? launch_route_gateup(a, *route, from_memory, s) : launch_gateup(a, from_memory, s)) return rc;
  return launch_down(a, from_memory, s);
}
