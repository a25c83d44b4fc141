// A small layer's down projection and combine in one launch: no y, no launch behind it.
//
// Replaces jax_gpt/models/qwen35/moe.py:87 (the third ragged_dot), :90-94 (_scatter_back), :225-232's last product and :281 for batches
// whose GEMMs read the selection themselves.  A workgroup owns 16 output columns of as many tokens as have 64 (or 128) selections,
// whatever their experts; a lane holds a selection (or two).  Selections of one expert find each other by ballots of the id's bits;
// every 16 of them are a unit of work, and so are 16 tokens of the shared expert.  A wave takes a unit through all of K in a ring of
// its own -- 16 weight rows and 8 or 16 rows of h, no barrier, no other wave's copies to wait for -- and leaves its rows, rounded to bf16, in
// LDS, where the workgroup adds a token's up in slot order.  The arithmetic of the grouped GEMM and the combine, instruction for
// instruction: the same bits.
//   What bounds it: a launch's start and its chain of dependent loads (ids, then rows and weights), then the bytes that a CU copies, some
// 70 a ns.  A unit copies 16 weight rows and 8 or 16 rows of h, whatever rows it has: some 240 KB a workgroup for 64 selections of 8
// experts of 512 x 1024, of which 192 KB are distinct.  A grouped GEMM has a work item for each 256 columns of an expert's rows, 40 of 288 KB on 256 CUs for
// 256 tokens of these.  That launch and the combine 8.6 + 3.1 us, this one 6.2; the call 22.9 -> 17.7 us, 384 tokens 23.5 -> 20.7, 512 25.6 ->
// 21.4; 32 experts of 1024 x 512 with a shared one, 64 tokens 24.5 -> 21.6.
//   Copies through LDS are what makes it: fragments loaded to registers are 64 bytes of each line, and the CU moves fewer bytes a ns
// (20.3 us for the 17.7, 27.7 for the 22 of 512 tokens).  Sixteen waves a workgroup with rings of two K steps.  Nothing that a wave waits for
// stands behind its copies: the unit's weight scales are copied in front of them.  With these in a register, whose first use in the K loop
// waited for all copies at every step, and 16 rows of h for every unit: a shared expert of 256 x 4096 beside 8 small ones, 64 tokens 22.8 us a
// call, so 18.6; tiny, 128 tokens 15.9 and 15.5.
#include "moe_small.h"

#include <math.h>

namespace {

constexpr int BK = 128, COLS = 16;   // output columns of a workgroup

constexpr int WAVES = 16, NST = 2;
constexpr int kMostSteps = 64;           // K steps (a lane copies the weight scale of one)

// LDS of a wave: NST stages of a K step, 16 weight rows and 16 rows of h with their scales (and 48 more), and the unit's weight scales
constexpr int kStage = 2 * 16 * BK + 256;
constexpr int kRing = NST * kStage, kWaveLds = kRing + kMostSteps * 4;

// PL: selections of a lane
template <int PL>
__global__ __launch_bounds__(64 * WAVES) void small_down_kernel(const SmallDown a, const int tokens) {
  constexpr int PAIRS = 64 * PL;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  __shared__ v4f y[2 * PAIRS][COLS / 4];   // rows of the selections, then of the shared expert
  __shared__ float weight[PAIRS];
  __shared__ int unit_rows[WAVES][16];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), fr = lane & 15, fq = lane >> 4;
  // XCD x has the column tiles x, x + 8, ...: its L2 holds an eighth of the weights, whatever the tokens
  const int per = a.D / (8 * COLS), i = blockIdx.x >> 3, group = i / per, ct = (i - group * per) * 8 + (blockIdx.x & 7);
  const int t0 = group * tokens, nt = min(tokens, a.M - t0), pairs = nt * a.k, p0 = t0 * a.k;
  int id[PL];
  bool valid[PL];
#pragma unroll
  for (int q = 0; q < PL; ++q) {
    const int p = q * 64 + lane;
    id[q] = p < pairs ? a.ids[p0 + p] : -1;
    valid[q] = (unsigned)id[q] < (unsigned)a.E;
  }
  // what the sums need, before the rest is under way
  constexpr int OUTS = (PAIRS * COLS + 64 * WAVES - 1) / (64 * WAVES);
  float residual[OUTS] = {}, gate[OUTS] = {};
#pragma unroll
  for (int o = 0; o < OUTS; ++o) {
    const int at = tid + o * 64 * WAVES, t = at / COLS;
    if (t < nt) {
      const size_t x = (size_t)(t0 + t) * a.D + ct * COLS + at % COLS;
      if (a.residual) residual[o] = bf16_to_f32(a.io_f32 ? f32_to_bf16(((const float*)a.residual)[x]) : ((const bf16_t*)a.residual)[x]);
      if (a.shared_gate) gate[o] = a.shared_gate[t0 + t];
    }
  }
  uint8_t* const ring = lds + w * kWaveLds;
  const unsigned ring_at = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)ring);
  if (tid < pairs) weight[tid] = a.w[p0 + tid];
  // each selection's place among those of its expert, and the first of every 16 of these: a unit
  int rank[PL] = {};
  unsigned long long leaders[PL], same[PL][PL];
#pragma unroll
  for (int r = 0; r < PL; ++r) {
#pragma unroll
    for (int q = 0; q < PL; ++q) same[q][r] = __ballot(valid[r]);
#pragma unroll
    for (int b = 0; b < 6; ++b) {
      const unsigned long long set = __ballot(id[r] >> b & 1);
#pragma unroll
      for (int q = 0; q < PL; ++q) same[q][r] &= id[q] >> b & 1 ? set : ~set;
    }
  }
  int routed = 0;
#pragma unroll
  for (int q = 0; q < PL; ++q) {
#pragma unroll
    for (int r = 0; r < q; ++r) rank[q] += (int)__popcll(same[q][r]);
    rank[q] += (int)__builtin_amdgcn_mbcnt_hi((unsigned)(same[q][q] >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)same[q][q], 0u));
    leaders[q] = __ballot(valid[q] && (rank[q] & 15) == 0);
    routed += (int)__popcll(leaders[q]);
    if (w == q && q * 64 + lane < pairs && !valid[q]) {   // a selection out of range has no row: zeros
#pragma unroll
      for (int c = 0; c < COLS / 4; ++c) y[q * 64 + lane][c] = (v4f){0.f, 0.f, 0.f, 0.f};
    }
  }
  const int units = routed + (a.SI ? (nt + 15) >> 4 : 0);
  auto skip_units = [&](int n) {
    for (int i = 0; i < n; ++i) {
      if (PL == 1 || leaders[0]) leaders[0] &= leaders[0] - 1;
      else leaders[PL - 1] &= leaders[PL - 1] - 1;
    }
  };
  skip_units(w);
  for (int u = w; u < units; u += WAVES) {
    const bool shared = u >= routed;
    int count, e = 0, first;   // rows of the unit
    if (shared) {
      first = (u - routed) * 16;
      count = min(16, nt - first);
    } else {
      const bool low = PL == 1 || leaders[0];
      const int at = (int)__builtin_ctzll(low ? leaders[0] : leaders[PL - 1]);
      skip_units(WAVES);
      e = __builtin_amdgcn_readlane(low ? id[0] : id[PL - 1], at);
      first = __builtin_amdgcn_readlane(low ? rank[0] : rank[PL - 1], at);
      count = 0;
#pragma unroll
      for (int q = 0; q < PL; ++q) {
        const bool mine = id[q] == e && (rank[q] & ~15) == first;
        count += (int)__popcll(__ballot(mine));
        if (mine) unit_rows[w][rank[q] & 15] = q * 64 + lane;
      }
      __builtin_amdgcn_wave_barrier();   // (within the wave: LDS operations stay in order)
    }
    const int K = shared ? a.SI : a.I, KB = K / BK;
    auto slot_of = [&](int r) { r = min(r, count - 1); return shared ? first + r : unit_rows[w][r]; };
    const int row0 = shared ? t0 : p0;
    const uint8_t* wp = (shared ? a.ws : a.wd) + ((size_t)e * a.D + ct * COLS) * K;
    const uint8_t* xp = (shared ? a.hsq : a.hq) + (size_t)row0 * K;
    const float* sx = (shared ? a.shs : a.sh) + (size_t)row0 * KB;
    const float* sw = (shared ? a.sws : a.swd) + ((size_t)e * (a.D / BK) + ct / 8) * KB;
    unsigned woff[2], xoff[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int r = g * 8 + (lane >> 3), piece = (lane & 7) ^ ((r >> 1) & 7);
      woff[g] = (unsigned)r * (unsigned)K + piece * 16;
      xoff[g] = (unsigned)slot_of(r) * (unsigned)K + piece * 16;
    }
    const unsigned soff = (unsigned)slot_of(fr) * (unsigned)KB * 4u;
    const bool wide = count > 8;
    auto copy = [&](int kb, int st) {
      const unsigned to = ring_at + st * kStage;
#pragma unroll
      for (int g = 0; g < 2; ++g) dma16(wp + (size_t)kb * BK, woff[g], to + g * 1024u);
      dma16(xp + (size_t)kb * BK, xoff[0], to + 2048u);
      if (wide) dma16(xp + (size_t)kb * BK, xoff[1], to + 3072u);
      dma4((const uint8_t*)(sx + kb), soff, to + 4096u);
    };
    // (copied too, in front of the first stage: a load to a register would be waited for with everything behind it)
    dma4((const uint8_t*)sw, (unsigned)min(lane, KB - 1) * 4u, ring_at + kRing);
    for (int t = 0; t < NST && t < KB; ++t) copy(t, t);
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    int st = 0;
    for (int kb = 0; kb < KB; ++kb) {
      if (KB - kb < NST) wait_vm<0>();
      else if (wide) wait_vm<5 * (NST - 1)>();
      else wait_vm<4 * (NST - 1)>();
      asm volatile("" ::: "memory");
      const uint8_t* base = ring + st * kStage;
      auto frag = [&](const uint8_t* p) {
        const v4i lo = *(const v4i*)(p + fr * BK + ((fq ^ (fr >> 1)) << 4)), hi = *(const v4i*)(p + fr * BK + (((fq + 4) ^ (fr >> 1)) << 4));
        return (v8i){lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      };
      const v8i wf = frag(base), xf = frag(base + 2048);
      const float c = ((const float*)(base + 4096))[fr] * ((const float*)(ring + kRing))[kb];
      if (kb + NST < KB) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the fragments are in registers: the stage may be overwritten
        copy(kb + NST, st);
      }
      st = st + 1 == NST ? 0 : st + 1;
      const v4f p = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf, xf, (v4f){0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
      acc += p * c;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (the next unit's copies overwrite the stages)
    const int slot = (shared ? PAIRS : 0) + slot_of(fr);
    __builtin_amdgcn_wave_barrier();
    if (fr < count) {   // the row in bf16
      const unsigned lo = pack2_bf16(acc[0], acc[1]), hi = pack2_bf16(acc[2], acc[3]);
      y[slot][fq] = (v4f){__uint_as_float(lo << 16), __uint_as_float(lo & 0xffff0000u), __uint_as_float(hi << 16), __uint_as_float(hi & 0xffff0000u)};
    }
  }
  __syncthreads();
#pragma unroll
  for (int o = 0; o < OUTS; ++o) {
#pragma clang fp contract(off)
    const int at = tid + o * 64 * WAVES, t = at / COLS, c = at % COLS;
    if (t >= nt) break;
    float s = 0.f;
    for (int j = t * a.k; j < (t + 1) * a.k; ++j) s = s + ((const float*)y[j])[c] * weight[j];
    if (a.SI) {
      const float v = ((const float*)y[PAIRS + t])[c];
      s = s + (a.shared_gate ? v * gate[o] : v);
    }
    if (a.residual) s = s + residual[o];
    const size_t x = (size_t)(t0 + t) * a.D + ct * COLS + c;
    const bf16_t r = f32_to_bf16(s);
    if (a.io_f32) ((float*)a.out)[x] = bf16_to_f32(r);
    else ((bf16_t*)a.out)[x] = r;
  }
}

}  // namespace

// A group of tokens reads every expert's rows that it has a selection of again, so this is for batches that one workgroup a CU covers,
// with 64 selections a workgroup or, where these are too many workgroups, with 128 (two of those on a CU are slower than 128: tiny, 384
// tokens 20.6 / 22.7 us, mini 256 24.8 / 29.3, tiny 700 as 704 of 64 or 352 of 128 29.2 / 28.7 for 26.2 of the three launches).
// Of these up to 500 KB of copies a workgroup, counted for an even routing: uneven ones have fewer units and gain more.  This way against
// three launches, even and uneven (normal offsets of 1 on the logits) routing, 8 to 64 experts of 256 to 2048 x 256 to 2048: with 64 selections
// up to 500 KB 0.74 to 0.99 and 0.74 to 0.92, up to 600 0.73 to 1.10 (64 experts of 256 x 512 1.02 to 1.09) and 0.75 to 0.97, up to 1000 0.81
// to 1.14 and 0.81 to 1.00; with 128 up to 500 0.82 to 1.01 and 0.83 to 0.95, up to 600 0.83 to 1.01 and 0.81 to 1.00, up to 1000 0.86 to 1.19
// and 0.84 to 1.05.
int moe_small_down_lanes(int M, int D, int E, int k, int I, int SI) {
  if (M < 1 || E > 64 || k < 1 || k > 32 || I > kMostSteps * BK || SI > kMostSteps * BK) return 0;
  for (int lanes = 1; lanes <= 2; ++lanes) {
    const int tokens = 64 * lanes / k, most = tokens < M ? tokens : M;
    if ((long long)((M + tokens - 1) / tokens) * (D / COLS) > 256) continue;
    const double touched = E * (1.0 - pow(1.0 - 1.0 / E, most * k)), rows = most * k / touched;   // experts, and rows of each
    // a K step's KB of units of 16 rows: weights and scales, and h eight rows at a time
    auto step = [](double rows) { return 2.25 * ceil(rows / 16 - 1e-9) + ceil(rows / 8 - 1e-9); };
    return touched * step(rows) * (I / BK) + step(most) * (SI / BK) <= 500 ? lanes : 0;
  }
  return 0;
}

namespace {
template <int PL> int launch(const SmallDown& a, hipStream_t s) {
  static std::atomic<unsigned long long> raised = {};
  const int tokens = 64 * PL / a.k, groups = (a.M + tokens - 1) / tokens, lds = WAVES * kWaveLds;
  if (int rc = moe_raise_lds_limit((const void*)small_down_kernel<PL>, lds, raised)) return rc;
  hipLaunchKernelGGL(small_down_kernel<PL>, dim3((unsigned)groups * (a.D / COLS)), dim3(64 * WAVES), lds, s, a, tokens);
  return moe_check_hip(hipGetLastError(), "small layer's down launch");
}
}  // namespace
int moe_small_down(const SmallDown& a, int lanes, moe_stream_t stream) {
  return lanes == 1 ? launch<1>(a, (hipStream_t)stream) : launch<2>(a, (hipStream_t)stream);
}
