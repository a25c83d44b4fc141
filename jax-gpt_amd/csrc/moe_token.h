// The experts of single tokens (moe_token.hip).
#pragma once
#include "moe_common.h"

constexpr int MOE_TOKEN_ROWS = 16;    // tokens
constexpr int MOE_TOKEN_SLOTS = 33;   // k <= 32 and the shared expert

struct TokenExperts {   // (E, N, K) codes and block scales
  const uint8_t *w_gate, *w_up, *w_down;
  const float *s_gate, *s_up, *s_down;
};
struct TokenArgs {
  const uint8_t* xq;   // (M, D) codes and their (M, D / 128) scales
  const float* sx;
  const int32_t* idx;  // (M, k)
  const float* w;
  TokenExperts routed, shared;
  int M, D, E, k, I, SI;   // (SI 0: no shared expert)
  float* h;                // (M, k + 1, h_stride) f32
  int h_stride;            // the wider of I and SI
  const float* shared_gate;
  const void* residual;
  int io_f32;              // of residual and out
  void* out;
};
// whether a call of M tokens takes this route
bool moe_token_takes(int M, int D, int E, int k, int I, int SI);
// the second launch: tiles of 16 output columns and waves of a workgroup, LDS of a wave
struct TokenDownPlan { int tiles, waves, wave_lds; };
TokenDownPlan moe_token_down_plan(int M, int D, int k, int I, int SI);
// K steps of a ring's stage in the two launches: 1 or 2
struct TokenStages { int gateup, down; };
TokenStages moe_token_stages(int M, int D, int k, int I, int SI, bool from_memory);
// whether the first launch routes and quantises the tokens too: from ready logits (or a given selection) and (M, D) bf16 activations,
// or behind a router that moe_front_takes
// (chain: dependent steps of one token's selection)
int moe_token_chain(int routing, int E, int k, int n_group, int topk_group);
bool moe_token_routes(int M, int D, int E, int k, int I, int SI, bool selected, int chain = 0);
bool moe_token_fronts(int M, int k, int I, int SI, bool norm, bool from_memory, int router = 0);   // router: its weights (columns x D)
struct TokenRoute {   // (checked: moe_route_check, moe_front_check)
  int routing;
  RouteArgs args;   // args.idx, args.w: the TokenArgs' own
  const void* x;
  const FrontArgs* front;   // null: ready logits, or
  bool selected;            // nothing to route
};
int moe_token_experts(const TokenArgs& a, bool from_memory, const TokenRoute* route, moe_stream_t stream);   // route: null, or such a call's
