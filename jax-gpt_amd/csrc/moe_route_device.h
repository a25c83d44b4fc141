// One token's routing by one wave, as device functions: of the routing launches (moe_route.hip) and of the launch that routes
// single tokens in front of their experts (moe_token.hip).  Files that include this are compiled with -ffp-contract=off: every
// operation is rounded by itself.
#pragma once
#include "moe_common.h"

namespace {

// 32-bit keys: larger key = larger value (-0 equals +0); 0 = absent
__device__ __forceinline__ unsigned make_key(float v) {
  const unsigned u = __float_as_uint(v + 0.0f);  // -0 -> +0
  return max((u & 0x80000000u) ? ~u : (u | 0x80000000u), 1u);   // (a NaN of all ones is still present)
}
__device__ __forceinline__ float key_value(unsigned u) {
  return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}

// Lane permutations inside a row of 16 lanes (DPP, a few cycles each): xor 1, xor 2, mirror of 8, mirror of 16 -- a
// maximum does not care which partner it meets, only that the set closes.  Reductions over ds_bpermute cost about
// 100 cycles per step, and routing is a chain of reductions.
template <int CTRL> __device__ __forceinline__ unsigned dpp(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, 0xF, 0xF, false);
}
constexpr int DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E, DPP_MIRROR8 = 0x141, DPP_MIRROR16 = 0x140, DPP_ROR4 = 0x124, DPP_ROR8 = 0x128;

// wave-wide maximum, as a scalar: row maxima by DPP, the four rows as scalars
__device__ __forceinline__ unsigned wave_max(unsigned k) {
  k = max(k, dpp<DPP_XOR1>(k));
  k = max(k, dpp<DPP_XOR2>(k));
  k = max(k, dpp<DPP_MIRROR8>(k));
  k = max(k, dpp<DPP_MIRROR16>(k));
  const unsigned a = (unsigned)__builtin_amdgcn_readlane((int)k, 0), b = (unsigned)__builtin_amdgcn_readlane((int)k, 16);
  const unsigned c = (unsigned)__builtin_amdgcn_readlane((int)k, 32), d = (unsigned)__builtin_amdgcn_readlane((int)k, 48);
  return max(max(a, b), max(c, d));
}
// The two largest of a set of keys, equal ones counted: meet() joins disjoint sets.
struct TwoBest {
  unsigned m1 = 0u, m2 = 0u;
  __device__ __forceinline__ void meet(unsigned o1, unsigned o2) {
    m2 = max(min(m1, o1), max(m2, o2));
    m1 = max(m1, o1);
  }
  template <int CTRL> __device__ __forceinline__ void meet_dpp() { meet(dpp<CTRL>(m1), dpp<CTRL>(m2)); }
  __device__ __forceinline__ void meet_wave() {   // of all lanes' sets, as scalars
    meet_dpp<DPP_XOR1>();
    meet_dpp<DPP_XOR2>();
    meet_dpp<DPP_MIRROR8>();
    meet_dpp<DPP_MIRROR16>();
    const unsigned r1 = m1, r2 = m2;
    m1 = m2 = 0u;
#pragma unroll
    for (int row = 0; row < 64; row += 16)
      meet((unsigned)__builtin_amdgcn_readlane((int)r1, row), (unsigned)__builtin_amdgcn_readlane((int)r2, row));
  }
};
// wave-wide sum in the pairing of a butterfly (partner lane ^ 32, 16, 8, 4, 2, 1), which fixes the rounding.  After the
// step over 8 lanes i and i ^ 8 hold the same value, so a rotation by 4 meets what lane ^ 4 holds.
__device__ __forceinline__ float wave_sum_f32(float v) {
  v = __fadd_rn(v, __shfl_xor(v, 32, MOE_WAVE));
  v = __fadd_rn(v, __shfl_xor(v, 16, MOE_WAVE));
  v = __fadd_rn(v, __uint_as_float(dpp<DPP_ROR8>(__float_as_uint(v))));
  v = __fadd_rn(v, __uint_as_float(dpp<DPP_ROR4>(__float_as_uint(v))));
  v = __fadd_rn(v, __uint_as_float(dpp<DPP_XOR2>(__float_as_uint(v))));
  v = __fadd_rn(v, __uint_as_float(dpp<DPP_XOR1>(__float_as_uint(v))));
  return v;
}
__device__ __forceinline__ float lane_f32(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// the k best of the wave's keys in order, ties to the lower index.  BLOCKED: element e lives in lane e / VPL, slot
// e % VPL; otherwise in lane e % 64, slot e / 64.  Lane i keeps the i-th: its index, key and (SCORES) score.
template <int VPL, bool BLOCKED, bool SCORES>
__device__ __forceinline__ void select_topk(unsigned (&key)[VPL], const float* score, int k, int& my_idx, unsigned& my_key,
                                            float& my_score) {
  const int lane = threadIdx.x & 63;
  for (int sel = 0; sel < k; ++sel) {
    unsigned local = key[0];
#pragma unroll
    for (int s = 1; s < VPL; ++s) local = max(local, key[s]);
    const unsigned best = wave_max(local);
    int owner = 0, slot = 0;
    if (BLOCKED) {
      owner = (int)__builtin_ctzll(__ballot(local == best));
#pragma unroll
      for (int s = VPL - 1; s >= 0; --s)
        if ((unsigned)__builtin_amdgcn_readlane((int)key[s], owner) == best) slot = s;
    } else {
#pragma unroll
      for (int s = VPL - 1; s >= 0; --s) {
        const unsigned long long in = __ballot(key[s] == best);
        if (in) owner = (int)__builtin_ctzll(in), slot = s;
      }
    }
    float sv = 0.f;
#pragma unroll
    for (int s = 0; s < VPL; ++s) {
      if (SCORES) {
        const float v = lane_f32(score[s], owner);
        sv = s == slot ? v : sv;
      }
      if (s == slot && lane == owner) key[s] = 0u;
    }
    if (lane == sel) {
      my_idx = BLOCKED ? owner * VPL + slot : owner + 64 * slot;
      my_key = best;
      my_score = sv;
    }
  }
}
// sum of the first k lanes' values in lane order
__device__ __forceinline__ float sum_first(float v, int k) {
  float s = 0.f;
  for (int i = 0; i < k; ++i) s = __fadd_rn(s, lane_f32(v, i));
  return s;
}

constexpr int ROUTE_SOFTMAX = MOE_ROUTING_SOFTMAX, ROUTE_GROUPED = MOE_ROUTING_SIGMOID_GROUPED;

// One token's selection by one wave.  row: its logits (global memory or LDS).  Lane < k gets its expert and
// weight, which are stored too with `store`.
struct Chosen {
  int expert;
  float weight;
};
template <int VPL>
__device__ __forceinline__ Chosen route_softmax_token(const RouteArgs& a, const float* row, int t, bool store = true) {
  const int lane = threadIdx.x & 63;
  float v[VPL];
  unsigned key[VPL], top = 0u;
#pragma unroll
  for (int s = 0; s < VPL; ++s) {
    const int e = lane + 64 * s;
    v[s] = e < a.E ? row[e] : -INFINITY;
    key[s] = e < a.E ? make_key(v[s]) : 0u;
    top = max(top, v[s] == v[s] ? key[s] : 0u);   // (a NaN ranks like any other value but is nobody's maximum: see below)
  }
  // A NaN logit counts as exp_det's lower end and leaves the other experts' weights alone; as the maximum it would make
  // every difference a NaN, every exponential that lower end, and all k weights equal.
  const float mx = key_value(wave_max(top));
  float part = 0.f;
#pragma unroll
  for (int s = 0; s < VPL; ++s)
    if (lane + 64 * s < a.E) part = __fadd_rn(part, exp_det(__fsub_rn(v[s], mx)));
  const float denom = wave_sum_f32(part);
  int my_idx = 0;
  unsigned my_key = 0u;
  float unused;
  select_topk<VPL, false, false>(key, nullptr, a.k, my_idx, my_key, unused);
  const float p = __fdiv_rn(exp_det(__fsub_rn(key_value(my_key), mx)), denom);
  const float psum = sum_first(p, a.k);
  const float weight = a.renorm ? __fdiv_rn(p, psum) : p;
  if (store && lane < a.k) {
    a.idx[(size_t)t * a.k + lane] = my_idx;
    a.w[(size_t)t * a.k + lane] = weight;
  }
  return {my_idx, weight};
}

template <int VPL>
__device__ __forceinline__ Chosen route_grouped_token(const RouteArgs& a, const float* row, int t, bool store = true) {
  const int lane = threadIdx.x & 63, E = a.E, n_group = a.n_group;
  float score[VPL];
  unsigned key[VPL];
#pragma unroll
  for (int s = 0; s < VPL; ++s) {
    const int e = lane * VPL + s;
    const bool ok = e < E;
    score[s] = ok ? sigmoid_det(row[e]) : 0.f;
    const float choice = __fadd_rn(score[s], (ok && a.bias) ? a.bias[e] : 0.f);
    key[s] = ok ? make_key(choice) : 0u;
  }
  if (a.topk_group < n_group) {
    // group score = sum of the two best choice scores of the group; a group is kept if fewer than topk_group of the
    // groups score higher (ties: lower index)
    const int per = E / n_group, lpg = per / VPL;   // experts and lanes per group
    if (lpg * VPL == per && (lpg & (lpg - 1)) == 0 && lpg >= 1 && lpg <= 16 && per >= 2) {
      // every group is a run of 1, 2, 4, 8 or 16 lanes: all groups' two best at once, by DPP
      TwoBest best;
#pragma unroll
      for (int s = 0; s < VPL; ++s) best.meet(key[s], 0u);
      if (lpg > 1) best.meet_dpp<DPP_XOR1>();
      if (lpg > 2) best.meet_dpp<DPP_XOR2>();
      if (lpg > 4) best.meet_dpp<DPP_MIRROR8>();
      if (lpg > 8) best.meet_dpp<DPP_MIRROR16>();
      const int g = lane / lpg;
      const unsigned gkey = make_key(__fadd_rn(key_value(best.m1), key_value(best.m2)));
      int rank = 0;
      for (int o = 0; o < n_group; ++o) {
        const unsigned ok = (unsigned)__builtin_amdgcn_readlane((int)gkey, o * lpg);
        rank += (ok > gkey || (ok == gkey && o < g)) ? 1 : 0;
      }
      const bool keep = rank < a.topk_group;
#pragma unroll
      for (int s = 0; s < VPL; ++s) key[s] = keep ? key[s] : 0u;
    } else {
      // groups that lie across lanes in any way: one at a time (lane g keeps group g's score).  (The second best as a
      // second maximum over what lies below the first, with a count of the equals: 8192 tokens of 640 experts in 4
      // groups 52 us, 46 this way.)
      unsigned gkey = 0u;
      int gid[VPL];
#pragma unroll
      for (int s = 0; s < VPL; ++s) gid[s] = lane * VPL + s < E ? (lane * VPL + s) / per : -1;
      for (int g = 0; g < n_group; ++g) {
        TwoBest best;
#pragma unroll
        for (int s = 0; s < VPL; ++s) best.meet(gid[s] == g ? key[s] : 0u, 0u);
        best.meet_wave();
        float gs = key_value(best.m1);
        if (per >= 2) gs = __fadd_rn(gs, key_value(best.m2));
        if (lane == g) gkey = make_key(gs);
      }
      int rank = 0;
      for (int o = 0; o < n_group; ++o) {
        const unsigned ok = (unsigned)__builtin_amdgcn_readlane((int)gkey, o);
        rank += (ok > gkey || (ok == gkey && o < lane)) ? 1 : 0;
      }
      const unsigned long long keep = __ballot(lane < n_group && rank < a.topk_group);   // bit g set = group g kept
#pragma unroll
      for (int s = 0; s < VPL; ++s)
        if (gid[s] < 0 || !((keep >> gid[s]) & 1ull)) key[s] = 0u;
    }
  }
  int my_idx = 0;
  unsigned my_key = 0u;
  float my_w = 0.f;
  select_topk<VPL, true, true>(key, score, a.k, my_idx, my_key, my_w);
  const float wsum = sum_first(my_w, a.k);
  const float weight = __fmul_rn(a.renorm ? __fdiv_rn(my_w, __fadd_rn(wsum, 1e-20f)) : my_w, a.routed_scale);
  if (store && lane < a.k) {
    a.idx[(size_t)t * a.k + lane] = my_idx;
    a.w[(size_t)t * a.k + lane] = weight;
  }
  return {my_idx, weight};
}

}  // namespace
