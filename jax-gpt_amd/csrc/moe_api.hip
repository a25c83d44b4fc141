// Error reporting and the whole-path entry point of the C ABI.
//
// moe_forward = jax_gpt/models/qwen35/moe.py:97-114 (expert_forward_single) fed by
// router logits, plus the shared expert of moe.py:225-232 and the add of :281.
#include <stdarg.h>
#include <stdio.h>

#include <mutex>

#include "moe_common.h"
#include "moe_small.h"
#include "moe_token.h"

static thread_local char g_err[512] = "";

int moe_set_error(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int moe_check_hip(hipError_t e, const char* what) {
  if (e == hipSuccess) return MOE_OK;
  return moe_set_error(MOE_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
}

extern "C" int moe_abi_version(void) { return 7; }
extern "C" const char* moe_last_error(void) { return g_err; }

namespace {

// One side stream per device, default priority, created on first use and kept for the life of the process.
int side_stream(hipStream_t* out) {
  static std::mutex mu;
  static hipStream_t streams[64] = {};
  int dev = 0;
  int rc = moe_check_hip(hipGetDevice(&dev), "forward: hipGetDevice");
  if (rc) return rc;
  if (dev < 0 || dev >= 64) return moe_set_error(MOE_ERR_HIP, "forward: device index %d out of range", dev);
  std::lock_guard<std::mutex> lock(mu);
  if (!streams[dev]) {
    if ((rc = moe_check_hip(hipStreamCreateWithFlags(&streams[dev], hipStreamNonBlocking), "forward: side stream")))
      return rc;
  }
  *out = streams[dev];
  return MOE_OK;
}

// The events of a call with a shared expert (fork, activations quantised, join), kept per host thread and device
// and created on first use: a call enqueues and returns on one thread, and a wait that is already enqueued keeps
// the record it was enqueued after, so the thread's next call may record the same events again (calls of other
// threads have their own).  They are never destroyed: the runtime may be gone by the time a thread ends.
struct CallEvents {
  hipEvent_t fork, quant, join;
};
int call_events(CallEvents** out) {
  static thread_local CallEvents events[64] = {};
  int dev = 0;
  int rc = moe_check_hip(hipGetDevice(&dev), "forward: hipGetDevice");
  if (rc) return rc;
  if (dev < 0 || dev >= 64) return moe_set_error(MOE_ERR_HIP, "forward: device index %d out of range", dev);
  CallEvents& ev = events[dev];
  if (!ev.join) {
    hipEvent_t made[3] = {};
    for (int i = 0; i < 3; ++i) {
      const hipError_t e = hipEventCreateWithFlags(&made[i], hipEventDisableTiming);
      if (e != hipSuccess) {
        for (int j = 0; j < i; ++j) (void)hipEventDestroy(made[j]);
        return moe_check_hip(e, "forward: creating the fork/join events");
      }
    }
    ev = CallEvents{made[0], made[1], made[2]};
  }
  *out = &ev;
  return MOE_OK;
}

struct Carver {
  char* base;
  size_t used;
  void* take(size_t bytes) {
    void* p = base ? base + used : nullptr;
    used += (bytes + 255) & ~(size_t)255;
    return p;
  }
};

struct ForwardBuffers {
  int32_t *idx, *group_sizes, *group_offsets, *sorted_token_ids, *inv_perm;
  float *h32, *w, *sx, *sh, *shs, *shared_gate, *sx_listed, *sx_blocked;
  uint8_t *xq, *hq, *hsq;
  void *y, *ys, *permute_ws, *gemm_ws, *gemm_down_ws, *router_ws, *normed;
  size_t permute_ws_bytes, gemm_ws_bytes, router_ws_bytes, total;
};

ForwardBuffers carve(void* ws, int M, int D, int E, int k, int I, int SI, bool router) {
  ForwardBuffers b;
  Carver c{(char*)ws, 0};
  const size_t R = (size_t)M * k;
  b.idx = (int32_t*)c.take(R * 4);
  b.w = (float*)c.take(R * 4);
  b.group_sizes = (int32_t*)c.take((size_t)E * 4);
  b.group_offsets = (int32_t*)c.take((size_t)(E + 1) * 4);
  b.sorted_token_ids = (int32_t*)c.take(R * 4);
  b.inv_perm = (int32_t*)c.take(R * 4);
  b.permute_ws_bytes = moe_permute_workspace_bytes(M, k, E);
  b.permute_ws = c.take(b.permute_ws_bytes);
  b.gemm_ws_bytes = moe_gemm_workspace_bytes((int)R, E, I > D ? I : D);
  b.gemm_ws = c.take(b.gemm_ws_bytes);   // tile list of the routed GEMMs
  b.xq = (uint8_t*)c.take((size_t)M * D);
  b.sx = (float*)c.take((size_t)M * (D / 128) * 4);
  // block-major copies of the activation scales for large batches (GemmScales): routed rows in sorted order,
  // and the tokens in their own order for the shared expert
  b.sx_listed = (float*)c.take(R * (D / 128) * 4);
  b.sx_blocked = SI ? (float*)c.take((size_t)M * (D / 128) * 4) : nullptr;
  b.hq = (uint8_t*)c.take(R * I);
  b.sh = (float*)c.take(R * (I / 128) * 4);
  b.y = c.take(R * D * 2);
  b.hsq = SI ? (uint8_t*)c.take((size_t)M * SI) : nullptr;
  b.shs = SI ? (float*)c.take((size_t)M * (SI / 128) * 4) : nullptr;
  b.ys = SI ? c.take((size_t)M * D * 2) : nullptr;
  b.shared_gate = router ? (float*)c.take((size_t)M * 4) : nullptr;
  const size_t few = M < MOE_TOKEN_ROWS ? M : MOE_TOKEN_ROWS;
  b.h32 = (float*)c.take(few * (k + 1) * (I > SI ? I : SI) * 4);   // h of single tokens
  b.router_ws_bytes = router ? moe_router_workspace_bytes(M, D, E) : 0;
  // The router's sums and, once the routing launch has added them up, the down GEMM's own list, if it has one (lists of several chunks: the
  // placing launch that writes them stands behind the routing launch).
  const size_t down_list = R > kSmallRows ? b.gemm_ws_bytes : 0;
  b.router_ws = b.gemm_down_ws = router ? c.take(b.router_ws_bytes > down_list ? b.router_ws_bytes : down_list) : nullptr;
  b.normed = router ? c.take((size_t)M * D * 2) : nullptr;   // RMS-normalised activations (norm_weight)
  b.total = c.used;
  return b;
}

}  // namespace

namespace {
// The activations that the router's matmul and the experts compute from: x itself, its RMS-normalised form or, from f32
// input, its bf16 rounding; the latter two are kept in b.normed for the matmul.
// (sx_blocked: an optional second copy of the scales, block-major in token order, for the shared expert of a large batch)
bool quantiser_feeds_router(const MoeForwardArgs* a, int io_f32) { return a->norm_weight || (io_f32 && a->w_router); }
int quantise(const MoeForwardArgs* a, int io_f32, const ForwardBuffers& b, float* sx_blocked, moe_stream_t stream) {
  if (a->norm_weight)
    return moe_rmsnorm_quant_impl(a->x, io_f32, a->norm_weight, a->norm_eps, a->M, a->D, b.normed, b.xq, b.sx, sx_blocked, stream);
  return moe_quant_act_impl(a->x, io_f32, quantiser_feeds_router(a, io_f32) ? b.normed : nullptr, a->M, a->D, b.xq, b.sx, sx_blocked, stream);
}

// Whether a call with a shared expert runs it inside the routed launches (true) or on the side stream.  The shared
// expert's GEMMs can fill the gap that quantising, routing and sorting leave in front of the routed ones, for the price
// of two streams' events.  Measured, together against forked: 4000 tokens of the mini layer 72 / 105 us, 2047 tokens of
// the Qwen3.5 layer 1269 / 1294 us, 4096 tokens 1456 / 1481; the DeepSeek-V3 layer at 777 tokens 1508 / 1513, at 2048
// 1975 / 1970, at 4096 2518 / 2505, at 8192 3847 / 3830 us.
bool small_batch(int M, int D) { return (long long)M * D <= (1ll << 24); }
}  // namespace

extern "C" size_t moe_forward_workspace_bytes(int M, int D, int E, int k, int I, int SI) {
  if (M < 0 || D <= 0 || E <= 0 || k <= 0 || I <= 0 || SI < 0) return 0;
  return carve(nullptr, M, D, E, k, I, SI, true).total;   // room for the router whether or not a call uses it
}

// given_idx / given_w: a selection that the caller has made (no routing), or null
static int forward(const MoeForwardArgs* a, int io_f32, const int32_t* given_idx, const float* given_w, void* ws, size_t ws_bytes, moe_stream_t stream) {
  MOE_REQUIRE(a && ws, MOE_ERR_NULL, "forward: null args or workspace");
  MOE_REQUIRE(a->M >= 0 && a->D > 0 && a->E >= 1 && a->k >= 1 && a->I > 0 && a->SI >= 0, MOE_ERR_BAD_SHAPE,
              "forward: bad dims M=%d D=%d E=%d k=%d I=%d SI=%d", a->M, a->D, a->E, a->k, a->I, a->SI);
  MOE_REQUIRE(a->D % 128 == 0 && a->I % 128 == 0 && a->SI % 128 == 0, MOE_ERR_BAD_SHAPE,
              "forward: D=%d, I=%d and SI=%d must be multiples of 128", a->D, a->I, a->SI);
  MOE_REQUIRE((a->M == 0 || (a->x && (a->logits || a->w_router || given_idx) && a->out)) && a->w_gate && a->w_up && a->w_down && a->sw_gate && a->sw_up && a->sw_down,
              MOE_ERR_NULL, "forward: null tensor pointer");
  if (a->SI)
    MOE_REQUIRE(a->ws_gate && a->ws_up && a->ws_down && a->sws_gate && a->sws_up && a->sws_down, MOE_ERR_NULL,
                "forward: SI > 0 but a shared-expert pointer is null");
  MOE_REQUIRE(MOE_ALIGNED16(ws), MOE_ERR_BAD_ALIGN, "forward: workspace must be 16-byte aligned");
  const size_t need = moe_forward_workspace_bytes(a->M, a->D, a->E, a->k, a->I, a->SI);
  MOE_REQUIRE(ws_bytes >= need, MOE_ERR_WORKSPACE_TOO_SMALL, "forward: workspace %zu < %zu", ws_bytes, need);
  if (a->M == 0) return MOE_OK;

  MOE_REQUIRE(!a->w_shared_gate || (a->w_router && a->SI), MOE_ERR_NULL,
              "forward: w_shared_gate needs w_router and a shared expert");
  MOE_REQUIRE(a->w_router || !a->out_logits, MOE_ERR_NULL, "forward: out_logits is an output of the router (w_router)");
  MOE_REQUIRE(a->w_shared_gate || !a->out_shared_gate, MOE_ERR_NULL, "forward: out_shared_gate needs w_shared_gate");
  ForwardBuffers b = carve(ws, a->M, a->D, a->E, a->k, a->I, a->SI, true);
  int32_t* idx = a->out_idx ? a->out_idx : b.idx;
  float* w_own = a->out_w ? a->out_w : b.w;
  const float* w = given_idx ? given_w : w_own;
  int32_t* gsz = a->out_group_sizes ? a->out_group_sizes : b.group_sizes;
  int32_t* stid = a->out_sorted_token_ids ? a->out_sorted_token_ids : b.sorted_token_ids;
  int32_t* inv = a->out_inv_perm ? a->out_inv_perm : b.inv_perm;
  // the intermediate h is written straight into the caller's debug arrays when both are given
  MOE_REQUIRE((a->out_hq == nullptr) == (a->out_sh == nullptr), MOE_ERR_NULL, "forward: out_hq and out_sh come together");
  MOE_REQUIRE(MOE_ALIGNED16(a->out_hq), MOE_ERR_BAD_ALIGN, "forward: out_hq must be 16-byte aligned");
  uint8_t* hq = a->out_hq ? a->out_hq : b.hq;
  float* sh = a->out_sh ? a->out_sh : b.sh;
  MOE_REQUIRE((a->out_hsq == nullptr) == (a->out_shs == nullptr) && (!a->out_hsq || a->SI), MOE_ERR_NULL,
              "forward: out_hsq and out_shs come together and need a shared expert");
  MOE_REQUIRE(MOE_ALIGNED16(a->out_hsq), MOE_ERR_BAD_ALIGN, "forward: out_hsq must be 16-byte aligned");
  uint8_t* hsq = a->out_hsq ? a->out_hsq : b.hsq;
  float* shs = a->out_shs ? a->out_shs : b.shs;
  MOE_REQUIRE(!a->out_ys || a->SI, MOE_ERR_NULL, "forward: out_ys needs a shared expert");
  MOE_REQUIRE(MOE_ALIGNED16(a->out_y) && MOE_ALIGNED16(a->out_ys), MOE_ERR_BAD_ALIGN, "forward: out_y / out_ys must be 16-byte aligned");
  void* y = a->out_y ? a->out_y : b.y;
  void* ys = a->out_ys ? a->out_ys : b.ys;
  const int R = a->M * a->k;
  // large batches read their activation scales from block-major arrays (GemmScales); a decode-sized batch touches
  // few scale lines either way and is spared the extra launch
  const bool blocked_scales = R > kSmallRows;
  hipStream_t main_s = (hipStream_t)stream;
  MOE_REQUIRE(given_idx || a->routing == MOE_ROUTING_SOFTMAX || a->routing == MOE_ROUTING_SIGMOID_GROUPED, MOE_ERR_BAD_SHAPE,
              "forward: unknown routing %d", a->routing);
  int rc;

  // The shared expert.  Small batches run it inside the routed experts' two GEMM launches: they are bound by launches
  // and by the host work behind them, and a second stream costs seven more of those (two events recorded and waited
  // for, three launches) where one more group of work items costs none: 1 token of the mini layer 97 -> 51 us, of the
  // DeepSeek-V3 layer 115 -> 100 us, 64 tokens of it 973 -> 965 us.
  //   Large batches fork at once: the side stream quantises the activations and runs the shared expert while the
  // caller's stream routes and permutes; the routed gate/up GEMM waits for the quantised activations, the combine for
  // the shared expert's output.  (Event record / wait is also the pattern that a capturing caller's graph turns into
  // forks and joins.)
  const bool fork = a->SI && !small_batch(a->M, a->D);
  hipStream_t side = nullptr;
  CallEvents* ev = nullptr;
  int rc_shared = MOE_OK;
  bool quant_joined = !fork;
  DenseGemm shared_gateup{}, shared_down{};
  if (a->SI) {
    GemmScales sc = moe_row_major_scales(a->D, a->SI);
    const float* sx_shared = b.sx;
    if (blocked_scales) {   // (block-major scales in token order: written by the quantiser itself)
      sx_shared = b.sx_blocked;
      sc.in_row = 1, sc.in_kb = a->M, sc.in_listed = true;
      if (!a->out_shs) sc.out_row = 1, sc.out_cb = a->M;   // (a debug copy of the h scales keeps the documented layout)
    }
    shared_gateup = DenseGemm{{b.xq, sx_shared, nullptr, a->ws_gate, a->sws_gate, a->ws_up, a->sws_up, a->D, a->SI, hsq, shs, sc}, a->M};
    shared_down = DenseGemm{{hsq, shs, nullptr, a->ws_down, a->sws_down, nullptr, nullptr, a->SI, a->D, ys, nullptr,
                             GemmScales{sc.out_row, sc.out_cb, true, 0, 0}}, a->M};
  }
  float* sx_blocked = a->SI && blocked_scales ? b.sx_blocked : nullptr;
  // Where the quantiser would run on the caller's stream just ahead of the routing kernel, the routing launch
  // carries its blocks instead (QuantJob: the two are independent; one launch less and they overlap).  Not where the
  // router reads what the quantiser writes.
  const bool quant_in_route = !fork && !quantiser_feeds_router(a, io_f32);
  // A small router: norm, quantiser, router matmul and selection are one launch.
  const int n_cols = a->E + (a->w_shared_gate ? 1 : 0);
  const bool front = !fork && a->w_router && !given_idx && MOE_ALIGNED16(a->norm_weight) &&
                     moe_front_takes(a->M, a->D, a->E, n_cols, a->norm_weight, io_f32, true);
  // A few tokens behind an RMSNorm: norm, quantiser and router matmul are one launch, below.
  const bool norm_router = !front && !fork && !sx_blocked && a->norm_weight && a->w_router && !given_idx &&
                           moe_norm_router_takes(a->M, a->D, n_cols, io_f32);
  QuantJob quant_job{};
  if (norm_router || front) {
  } else if (quant_in_route) {
    if ((rc = moe_quant_act_job(a->x, io_f32, nullptr, a->M, a->D, b.xq, b.sx, sx_blocked, &quant_job))) return rc;
  } else if (!fork) {
    if ((rc = quantise(a, io_f32, b, sx_blocked, stream))) return rc;
  } else {
    if ((rc = side_stream(&side))) return rc;
    if ((rc = call_events(&ev))) return rc;
    hipError_t e = hipEventRecord(ev->fork, main_s);
    if (e == hipSuccess) e = hipStreamWaitEvent(side, ev->fork, 0);
    if (e != hipSuccess) return moe_check_hip(e, "forward: fork");
    rc_shared = quantise(a, io_f32, b, sx_blocked, (moe_stream_t)side);
    if (!rc_shared) rc_shared = moe_check_hip(hipEventRecord(ev->quant, side), "forward: quant event");
    if (!rc_shared) rc_shared = moe_gemm_gateup_impl(nullptr, &shared_gateup, (moe_stream_t)side);
    if (!rc_shared) rc_shared = moe_gemm_down_impl(nullptr, &shared_down, (moe_stream_t)side);
  }
  // Once the side stream has been forked off this call, the join is enqueued on every path out of here, so that the
  // caller's stream (or the graph it is being captured into) never loses track of the side stream.
  auto join = [&](int code) {
    if (!fork) return code;
    hipError_t e1 = hipEventRecord(ev->join, side);
    hipError_t e2 = hipStreamWaitEvent(main_s, ev->join, 0);
    if (code) return code;
    if (rc_shared) return rc_shared;
    if (e1 != hipSuccess) return moe_check_hip(e1, "forward: join");
    return moe_check_hip(e2, "forward: join");
  };

  // With a router weight the routing kernel adds the matmul's split-K partial sums itself: the (M, E) logits
  // are written only when out_logits asks for them.
  LogitSource src{a->logits, nullptr, 0, a->E, nullptr, nullptr};
  const float* shared_gate = nullptr;
  float* gate_out = a->out_shared_gate ? a->out_shared_gate : b.shared_gate;   // (written by the routing kernel)
  if (a->w_shared_gate && !given_idx) shared_gate = gate_out;
  if (front) {
    src = LogitSource{nullptr, nullptr, 0, n_cols, a->out_logits, gate_out};
  } else if (a->w_router && !given_idx) {
    const bool from_quantiser = quantiser_feeds_router(a, io_f32);
    if (from_quantiser && !quant_joined) {   // (the quantiser was forked)
      if (rc_shared) return join(rc_shared);
      if ((rc = moe_check_hip(hipStreamWaitEvent(main_s, ev->quant, 0), "forward: quant join"))) return join(rc);
      quant_joined = true;
    }
    int splits = 0, used_cols = 0;
    if (norm_router)
      rc = moe_norm_router_partials(a->x, io_f32, a->norm_weight, a->norm_eps, a->M, a->D, a->w_router, a->E, a->w_shared_gate,
                                    b.xq, b.sx, b.router_ws, b.router_ws_bytes, &splits, &used_cols, stream);
    else
      rc = moe_router_partials(from_quantiser ? b.normed : a->x, a->M, a->D, a->w_router, a->E, a->w_shared_gate,
                               b.router_ws, b.router_ws_bytes, &splits, &used_cols, stream);
    if (rc) return join(rc);
    src = LogitSource{nullptr, (const float*)b.router_ws, splits, used_cols, a->out_logits, gate_out};
  }
  const RouteArgs route{src, a->bias, a->M, a->E, a->k, a->renorm, a->n_group, a->topk_group, a->routed_scale, idx, w_own};
  const QuantJob* carried = quant_in_route && !front ? &quant_job : nullptr;
  const FrontArgs front_args{a->x, io_f32, a->D, a->norm_weight, a->norm_eps, a->w_router, a->w_shared_gate, b.xq, b.sx, sx_blocked};
  auto select = [&](const PermuteOut* sort) {
    return front ? moe_front_impl(a->routing, route, front_args, sort, b.permute_ws, b.permute_ws_bytes, stream)
                 : moe_route_impl(a->routing, route, carried, sort, b.permute_ws, b.permute_ws_bytes, stream);
  };
  // A few tokens whose sort and rows nobody asks for: the experts straight from the selection.  (What the launches that this
  // leaves out would have refused is refused here.)
  const bool sorted_outputs = a->out_group_sizes || a->out_sorted_token_ids || a->out_inv_perm || a->out_hq || a->out_hsq || a->out_y || a->out_ys;
  if (!fork && !sorted_outputs && moe_token_takes(a->M, a->D, a->E, a->k, a->I, a->SI)) {
    const GemmScales sc = moe_row_major_scales(a->D, a->I);
    if ((rc = moe_gemm_check(GemmOperands{b.xq, b.sx, nullptr, a->w_gate, a->sw_gate, a->w_up, a->sw_up, a->D, a->I, hq, sh, sc}, R, a->E, false))) return rc;
    if ((rc = moe_gemm_check(GemmOperands{hq, sh, nullptr, a->w_down, a->sw_down, nullptr, nullptr, a->I, a->D, y, nullptr, sc}, R, a->E, true))) return rc;
    if (a->SI && (rc = moe_gemm_check(shared_gateup.op, a->M, 1, false))) return rc;
    if (a->SI && (rc = moe_gemm_check(shared_down.op, a->M, 1, true))) return rc;
    MOE_REQUIRE(MOE_ALIGNED16(a->out) && (!a->add_residual || MOE_ALIGNED16(a->x)), MOE_ERR_BAD_ALIGN,
                "combine: pointers must be 16-byte aligned");
    const bool from_memory = moe_gemm_from_memory(((long long)a->E * a->I + a->SI) * a->D);
    const bool fronts = front && moe_token_fronts(a->M, a->k, a->I, a->SI, a->norm_weight, from_memory, n_cols * a->D);
    const int chain = given_idx ? 0 : moe_token_chain(a->routing, a->E, a->k, a->n_group, a->topk_group);
    const bool routes = carried && !a->w_router && !io_f32 && moe_token_routes(a->M, a->D, a->E, a->k, a->I, a->SI, given_idx, chain);
    TokenRoute tok_route{a->routing, route, a->x, fronts ? &front_args : nullptr, given_idx != nullptr};
    if (given_idx) rc = carried && !routes ? moe_quant_act_impl(a->x, io_f32, nullptr, a->M, a->D, b.xq, b.sx, nullptr, stream) : MOE_OK;
    else if (fronts) rc = moe_front_check(a->routing, tok_route.args, front_args, false);
    else rc = routes ? moe_route_check(a->routing, route) : select(nullptr);
    if (rc) return rc;
    const TokenArgs tok{b.xq, b.sx, given_idx ? given_idx : idx, w,
                        TokenExperts{a->w_gate, a->w_up, a->w_down, a->sw_gate, a->sw_up, a->sw_down},
                        TokenExperts{a->ws_gate, a->ws_up, a->ws_down, a->sws_gate, a->sws_up, a->sws_down},
                        a->M, a->D, a->E, a->k, a->I, a->SI, b.h32, a->I > a->SI ? a->I : a->SI,
                        shared_gate, a->add_residual ? a->x : nullptr, io_f32, a->out};
    return moe_token_experts(tok, from_memory, fronts || routes ? &tok_route : nullptr, stream);
  }
  // routing, the sort by expert and the routed GEMMs' work list (the sort holds every expert's row range anyway)
  TileList tiles;
  const bool together = a->SI && !fork;   // the shared expert runs inside the routed launches
  const TileShape shape{R, a->E, a->M, {a->I / 128, (a->D + 255) / 256}, {a->D / 128, a->I / 128},
                        together ? a->M : 0, {a->SI / 128, (a->D + 255) / 256}};
  const bool from_memory = moe_gemm_from_memory(((long long)a->E * a->I + (together ? a->SI : 0)) * a->D);
  if (const int scan_rows = fork || sorted_outputs ? 0 : moe_gemm_scan_rows(shape, from_memory)) {
    // a small layer's few rows: the GEMMs read the selection itself
    const int32_t* ids = given_idx ? given_idx : idx;
    if (given_idx) rc = carried ? moe_quant_act_impl(a->x, io_f32, nullptr, a->M, a->D, b.xq, b.sx, nullptr, stream) : MOE_OK;
    else rc = select(nullptr);
    if (rc) return rc;
    const GemmScales sc = moe_row_major_scales(a->D, a->I);
    const RoutedGemm gateup{{b.xq, b.sx, nullptr, a->w_gate, a->sw_gate, a->w_up, a->sw_up, a->D, a->I, hq, sh, sc},
                            nullptr, a->E, R, nullptr, 0, scan_rows, 0, ids, a->k};
    const RoutedGemm down{{hq, sh, nullptr, a->w_down, a->sw_down, nullptr, nullptr, a->I, a->D, y, nullptr, moe_row_major_scales(a->I, a->D)},
                          nullptr, a->E, R, nullptr, 0, scan_rows, 0, ids, a->k};
    if ((rc = moe_gemm_gateup_impl(&gateup, together ? &shared_gateup : nullptr, stream))) return rc;
    // (what the launches that this one replaces would have refused is refused here)
    if (const int lanes = moe_small_down_lanes(a->M, a->D, a->E, a->k, a->I, a->SI)) {
      if ((rc = moe_gemm_check(down.op, R, a->E, true))) return rc;
      if (together && (rc = moe_gemm_check(shared_down.op, a->M, 1, true))) return rc;
      MOE_REQUIRE(MOE_ALIGNED16(a->out) && (!a->add_residual || MOE_ALIGNED16(a->x)), MOE_ERR_BAD_ALIGN,
                  "combine: pointers must be 16-byte aligned");
      return moe_small_down(SmallDown{hq, a->w_down, sh, a->sw_down, hsq, a->ws_down, shs, a->sws_down, ids, w, shared_gate,
                                      a->add_residual ? a->x : nullptr, io_f32, a->out, a->M, a->D, a->E, a->k, a->I, a->SI}, lanes, stream);
    }
    if ((rc = moe_gemm_down_impl(&down, together ? &shared_down : nullptr, stream))) return rc;
    return moe_combine_impl(y, w, ids, a->E, a->SI ? ys : nullptr, shared_gate, a->add_residual ? a->x : nullptr, io_f32, a->M, a->k, a->D,
                            a->out, stream);
  }
  const int tile_rows = moe_gemm_tile_rows(shape);
  const int down_rows = moe_gemm_down_tile_rows(shape, tile_rows);
  TileList down_tiles{};
  if ((rc = moe_gemm_tile_list(R, a->E, tile_rows, a->I / 128, down_rows ? 0 : (a->D + 255) / 256,
                               (down_rows || a->D < a->I ? a->D : a->I) / 128, b.gemm_ws, b.gemm_ws_bytes, &tiles))) return join(rc);
  if (down_rows && (rc = moe_gemm_tile_list(R, a->E, down_rows, 0, (a->D + 255) / 256, a->I / 128, b.gemm_down_ws, b.gemm_ws_bytes, &down_tiles)))
    return join(rc);
  const ScalePlan plan = moe_scale_plan(R, a->E, a->D, a->I, fork);
  const ScaleGather gather{b.sx, a->D / 128, b.sx_listed};
  const PlaceMore more{down_rows ? &down_tiles : nullptr, plan.placed ? &gather : nullptr};
  const PermuteOut sort{gsz, b.group_offsets, stid, nullptr, inv, a->k, tiles, down_rows || plan.placed ? &more : nullptr};
  rc = given_idx ? moe_permute_impl(given_idx, a->M, a->k, a->E, sort, b.permute_ws, b.permute_ws_bytes, carried, stream)
                 : select(&sort);
  if (rc) return join(rc);
  if (!quant_joined) {
    if (rc_shared) return join(rc_shared);
    if ((rc = moe_check_hip(hipStreamWaitEvent(main_s, ev->quant, 0), "forward: quant join"))) return join(rc);
  }
  GemmScales sc = moe_row_major_scales(a->D, a->I);
  const float* sx_routed = b.sx;
  if (blocked_scales && !a->out_sh) sc.out_row = 1, sc.out_cb = R;
  if (plan.gathered) {
    if (!plan.placed && (rc = moe_gather_scales(b.sx, stid, R, a->D / 128, b.sx_listed, stream))) return join(rc);
    sx_routed = b.sx_listed;
    sc.in_row = 1, sc.in_kb = R, sc.in_listed = true;
  }
  const RoutedGemm routed_gateup{{b.xq, sx_routed, stid, a->w_gate, a->sw_gate, a->w_up, a->sw_up, a->D, a->I, hq, sh, sc},
                                 b.group_offsets, a->E, R, b.gemm_ws, b.gemm_ws_bytes, tile_rows, tiles.pool_tiles};
  const RoutedGemm routed_down{{hq, sh, nullptr, a->w_down, a->sw_down, nullptr, nullptr, a->I, a->D, y, nullptr,
                                GemmScales{sc.out_row, sc.out_cb, true, 0, 0}},
                               b.group_offsets, a->E, R, down_rows ? b.gemm_down_ws : b.gemm_ws, b.gemm_ws_bytes,
                               down_rows ? down_rows : tile_rows, down_rows ? down_tiles.pool_tiles : tiles.pool_tiles};
  if ((rc = moe_gemm_gateup_impl(&routed_gateup, together ? &shared_gateup : nullptr, stream))) return join(rc);
  if ((rc = moe_gemm_down_impl(&routed_down, together ? &shared_down : nullptr, stream))) return join(rc);
  if ((rc = join(MOE_OK))) return rc;
  return moe_combine_impl(y, w, inv, 0, a->SI ? ys : nullptr, shared_gate, a->add_residual ? a->x : nullptr, io_f32, a->M, a->k,
                          a->D, a->out, stream);
}

extern "C" int moe_forward(const MoeForwardArgs* a, void* ws, size_t ws_bytes, moe_stream_t stream) {
  return forward(a, 0, nullptr, nullptr, ws, ws_bytes, stream);
}
extern "C" int moe_forward_f32(const MoeForwardArgs* a, void* ws, size_t ws_bytes, moe_stream_t stream) {
  return forward(a, 1, nullptr, nullptr, ws, ws_bytes, stream);
}
extern "C" int moe_forward_selected(const MoeForwardArgs* a, const int32_t* idx, const float* w, void* ws, size_t ws_bytes,
                                    moe_stream_t stream) {
  MOE_REQUIRE(a && (a->M == 0 || (idx && w)), MOE_ERR_NULL, "forward: null selection");
  MOE_REQUIRE(!a->w_router && !a->w_shared_gate, MOE_ERR_NULL, "forward: a selection that is given leaves the router nothing to do");
  return forward(a, 0, idx, w, ws, ws_bytes, stream);
}
