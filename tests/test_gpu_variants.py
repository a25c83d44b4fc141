"""The kernels' variants against each other and against the oracle, at the sizes where the choice between them changes:
row-tile heights and cache policies of the grouped GEMM, the shared expert inside or beside the routed launches, the
one-launch sort, the remainders of the router's K slices, rows of the RMSNorm, f32 activations.

Where two variants do the same individually rounded operations in the same order, the results must be equal bit for bit;
a row's result does not depend on the tile that it is computed in (one scale block of K per matrix instruction, added in
K order)."""
import numpy as np
import pytest

from oracle import moe_oracle as O
from tests import helpers as H
from tests.test_gpu_parity import _check_logits, _ragged_case, jg, test_rmsnorm_quant_vs_oracle as check_rmsnorm, test_route_sigmoid_grouped_bit_exact as check_grouped  # noqa: F401

pytestmark = pytest.mark.gpu

HEIGHTS = [257, 288, 289, 1, 32, 33, 576, 577, 0, 97, 128, 129, 160, 161, 192, 224, 225, 256]


@pytest.mark.parametrize("E,D,I,sizes", [
    (96, 1024, 1024, HEIGHTS),    # 8 K steps: little more than the rings' depth
    (96, 512, 1024, HEIGHTS),     # weights that the memory-side cache holds: plain copies, tall gate/up tiles ...
    (96, 2048, 256, HEIGHTS),     # ... and tall down tiles, over 4 and 2 K steps
    (96, 2048, 1024, HEIGHTS),    # full tiles up to 288 rows; two tiles share their lines (K = 2048)
    (64, 2304, 1536, HEIGHTS),    # K above 2048: two tiles do not; the down GEMM has fewer items and shorter tiles
    (64, 2304, 2048, [1, 31, 32, 33, 40, 64, 65, 96, 97, 128]),   # a weight stream with outputs above 4 MB: written through
])
def test_row_tile_variants_give_the_same_bits(jg, E, D, I, sizes):
    import torch
    print("row tiles", E, D, I, flush=True)
    sizes = [sizes[i % len(sizes)] for i in range(E)]
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    R = int(off[-1])
    gen = torch.Generator(device="cuda")
    gen.manual_seed(D + I)
    rand = lambda *s: torch.randn(s, dtype=torch.bfloat16, device="cuda", generator=gen)
    ex = {n: jg.quantize_weight_block(rand(E, *s).mul_(0.02))
          for n, s in (("gate", (I, D)), ("up", (I, D)), ("down", (D, I)))}
    xq, sx = jg.quant_act(rand(R, D))
    doff = H.to_cuda(off)
    hq, sh = jg.gemm_gateup_swiglu(xq, sx, ex["gate"], ex["up"], doff)
    y = jg.gemm_down(hq, sh, ex["down"], doff)
    for e in range(len(HEIGHTS)):
        one = {n: {k: v[e:e + 1] for k, v in d.items()} for n, d in ex.items()}
        for lo in range(int(off[e]), int(off[e + 1]), 32):      # the same rows, 32 at a time
            hi = min(lo + 32, int(off[e + 1]))
            o1 = H.to_cuda(np.array([0, hi - lo], np.int32))
            hq1, sh1 = jg.gemm_gateup_swiglu(xq[lo:hi], sx[lo:hi].clone(), one["gate"], one["up"], o1)
            y1 = jg.gemm_down(hq[lo:hi], sh[lo:hi].clone(), one["down"], o1)
            assert torch.equal(hq1.view(torch.uint8), hq[lo:hi].view(torch.uint8)), f"expert {e}, row {lo}: h"
            assert torch.equal(sh1, sh[lo:hi]), f"expert {e}, row {lo}: scales of h"
            assert torch.equal(y1, y[lo:hi]), f"expert {e}, row {lo}: y"
        if sizes[e] in (33, 97):                                 # and against the oracle (the classes agree with each other)
            lo, hi = int(off[e]), int(off[e]) + 33
            w, s = one["down"]["w"], one["down"]["scale_inv"]
            want = O.grouped_gemm(H.codes_np(hq[lo:hi]), sh[lo:hi].cpu().numpy(), H.codes_np(w), s.cpu().numpy(), np.array([0, hi - lo], np.int32))
            H.assert_close_out(H.bf16_to_np(y[lo:hi]), O.bf16_round(want.astype(np.float32)))


def _layer(jg, D, E, I, SI, seed):
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    rand = lambda *s: torch.randn(s, dtype=torch.bfloat16, device="cuda", generator=gen)
    q = lambda *s: jg.quantize_weight_block(rand(*s).mul_(0.02))
    params = dict(gate_proj=q(E, I, D), up_proj=q(E, I, D), down_proj=q(E, D, I),
                  gate_weight=rand(E, D).mul_(0.02).t(), shared_expert_gate_weight=rand(1, D).mul_(0.02).t())
    if SI:
        params.update(shared_gate_proj=q(1, SI, D), shared_up_proj=q(1, SI, D), shared_down_proj=q(1, D, SI))
    return params, rand


def test_shared_expert_beside_the_routing_gives_the_bits_of_the_joint_launches(jg):
    """Above 16 M activation elements the shared expert runs on the side stream: same bits as a sub-batch that takes it
    into the routed launches, and as every replay of a captured graph."""
    import torch
    print("forked shared expert", flush=True)
    D, E, k = 4096, 8, 2
    params, rand = _layer(jg, D, E, 128, 256, 3)
    M = (1 << 24) // D + 40
    x, lg = rand(M, D), rand(M, E).float()
    kw = dict(top_k=k, experts={n: params[n] for n in ("gate_proj", "up_proj", "down_proj")},
              shared={n: params["shared_" + n] for n in ("gate_proj", "up_proj", "down_proj")})
    full = jg.moe_experts(x, lg, **kw)
    part = jg.moe_experts(x[:1000].contiguous(), lg[:1000].contiguous(), **kw)
    assert torch.equal(full[:1000], part)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = jg.moe_experts(x, lg, **kw)
    for i in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, full), f"replay {i}"
        assert torch.equal(jg.moe_experts(x, lg, **kw), full)


@pytest.mark.parametrize("SI", [256, 0])
def test_large_f32_activations_give_the_bits_of_their_bf16_rounding(jg, SI):
    """Above 16 M activation elements, with a shared expert: the quantiser on the side stream feeds the router, and the
    combine reads f32.  Eager, and every replay of a captured graph with eager calls between."""
    import torch
    print("large f32 activations", SI, flush=True)
    D, k = 4096, 2
    params, rand = _layer(jg, D, 8, 128, SI, 5)
    M = (1 << 24) // D + 41
    gen = torch.Generator(device="cuda")
    gen.manual_seed(6)
    x = torch.randn((1, M, D), device="cuda", generator=gen)
    norm = rand(D).float() * 0.1
    xb = x.to(torch.bfloat16)
    for call in (lambda v: jg.moe_layer(v, params, k), lambda v: jg.moe_sublayer(v, norm, params, k)):
        want = call(xb).float()
        assert torch.equal(call(x), want)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = call(x)
        for i in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want), f"replay {i}"
            assert torch.equal(call(x), want)


def test_large_layer_with_its_router_is_its_stages(jg):
    """The forked path with the router inside: its logits and gate are the router's own, its rows those of a smaller batch
    that runs the shared expert in the routed launches, its output their combine."""
    import torch
    print("large layer with its router", flush=True)
    D, k = 4096, 2
    params, rand = _layer(jg, D, 8, 128, 256, 7)
    x = rand((1 << 24) // D + 41, D)
    ex, sh = ({n: params[p + n] for n in ("gate_proj", "up_proj", "down_proj")} for p in ("", "shared_"))
    out, dbg = jg.moe_experts(x, None, top_k=k, experts=ex, shared=sh, gate_weight=params["gate_weight"],
                              shared_expert_gate_weight=params["shared_expert_gate_weight"], return_debug=True)
    logits, gate = jg.router_logits(x, params["gate_weight"], params["shared_expert_gate_weight"])
    assert torch.equal(dbg["logits"], logits) and torch.equal(dbg["shared_gate"], gate)
    idx, w = jg.route_softmax_topk(logits, k)
    assert torch.equal(dbg["indices"], idx) and torch.equal(dbg["weights"], w)
    _, part = jg.moe_experts(x[:1000].contiguous(), logits[:1000].contiguous(), top_k=k, experts=ex, shared=sh, return_debug=True)
    rows = lambda d: d["y"][d["inv_perm"][:1000 * k].long()]
    assert torch.equal(rows(dbg), rows(part)) and torch.equal(dbg["ys"][:1000], part["ys"])
    assert torch.equal(out, jg.combine(dbg["y"], w, dbg["inv_perm"], dbg["ys"], gate))
    assert torch.equal(jg.moe_layer(x[None], params, k)[0], out)      # (debug arrays keep h scales row-major)


@pytest.mark.parametrize("M", [5, 300, (1 << 24) // 4096 + 9])
def test_given_selection_with_a_shared_expert(jg, M):
    """moe_forward_selected beside a shared expert, in the routed launches and forked: the routed call's bits."""
    import torch
    from jax_gpt_amd import moe
    print("given selection with a shared expert", M, flush=True)
    D, k = 4096, 2
    params, rand = _layer(jg, D, 8, 128, 256, M)
    x, lg = rand(max(M, 40), D), rand(max(M, 40), 8).float()
    ex, sh = ({n: params[p + n] for n in ("gate_proj", "up_proj", "down_proj")} for p in ("", "shared_"))
    want = jg.moe_experts(x, lg, top_k=k, experts=ex, shared=sh)[:M]      # (five tokens go straight to their experts, forty do not)
    x, lg = x[:M], lg[:M]
    assert torch.equal(moe._forward(x, None, k, ex, shared=sh, selected=jg.route_softmax_topk(lg, k)), want)


@pytest.mark.parametrize("M,E,k,D", [
    (1, 32, 2, 128), (8, 40, 3, 384),        # routed and sorted in one launch; 1 and 3 K slices
    (9, 40, 3, 640), (8, 512, 10, 1152),     # one token more; 9 slices: a batch of eight and one
    (33, 1000, 32, 1536),                    # eight counting waves, 12 slices
    (70, 8, 2, 256), (2100, 33, 1, 1280),    # 3 waves of entries; several chunks, experts not a multiple of four
    (1100, 1024, 4, 256),
    (872, 300, 3, 128), (873, 300, 3, 128),  # counted for the sort by the routing launch, and by the sort's own
    (1024, 64, 3, 128), (1026, 64, 3, 128),  # a token per workgroup and four (two left over) where nothing is sorted
])
def test_routing_inside_the_layer_is_exact(jg, M, E, k, D):
    """Selection and sort against the oracle on the logits that the layer ranked, which are the router's own."""
    import torch
    print("routing", M, E, k, D, flush=True)
    params, rand = _layer(jg, D, E, 128, 0, M + E)
    x = rand(M, D)
    out, dbg = jg.moe_experts(x, None, top_k=k, experts={n: params[n] for n in ("gate_proj", "up_proj", "down_proj")},
                              gate_weight=params["gate_weight"], return_debug=True)
    logits = dbg["logits"].cpu().numpy()
    own = jg.router_logits(x, params["gate_weight"])
    own = own[0] if isinstance(own, tuple) else own
    assert np.array_equal(logits, own.cpu().numpy())
    xn, wn = H.bf16_to_np(x), H.bf16_to_np(params["gate_weight"])
    _check_logits(logits, O.router_logits(xn, wn), np.abs(xn).astype(np.float64) @ np.abs(wn).astype(np.float64))
    idx, w = O.route_softmax_topk(logits, k)
    assert np.array_equal(dbg["indices"].cpu().numpy(), idx)
    assert np.allclose(dbg["weights"].cpu().numpy(), w, rtol=2e-6, atol=1e-9)
    ref = O.sort_and_group(idx, E)
    for name in ("group_sizes", "sorted_token_ids", "inv_perm"):
        assert np.array_equal(dbg[name].cpu().numpy(), ref[name]), name
    # the reference's two functions one after the other: the same path behind a selection that is handed in
    sel = jg.moe_routing(x, params["gate_weight"], k)
    assert torch.equal(sel[0], dbg["indices"]) and torch.equal(sel[1], dbg["weights"])
    assert torch.equal(jg.expert_forward_single(x, *sel, params["gate_proj"], params["up_proj"], params["down_proj"]), out)


@pytest.mark.parametrize("M,E,k", [(9, 8, 2), (32, 8, 2), (33, 8, 2), (22, 40, 3), (17, 300, 4), (513, 512, 5), (2049, 513, 1)])
def test_ready_logits_routed_and_sorted_in_one_launch_or_two(jg, M, E, k):
    print("routing of ready logits", M, E, k, flush=True)
    params, rand = _layer(jg, 128, E, 128, 0, M)
    lg = rand(M, E).float()
    _, dbg = jg.moe_experts(rand(M, 128), lg, top_k=k, return_debug=True,
                            experts={n: params[n] for n in ("gate_proj", "up_proj", "down_proj")})
    idx, _ = O.route_softmax_topk(lg.cpu().numpy(), k)
    assert np.array_equal(dbg["indices"].cpu().numpy(), idx)
    ref = O.sort_and_group(idx, E)
    for name in ("group_sizes", "sorted_token_ids", "inv_perm"):
        assert np.array_equal(dbg[name].cpu().numpy(), ref[name]), name


@pytest.mark.parametrize("E,G,TG,k", [(60, 3, 2, 4), (300, 4, 2, 8), (640, 4, 1, 8), (1000, 10, 3, 32), (64, 64, 5, 5), (1024, 2, 1, 6), (130, 13, 4, 7)])
def test_groups_across_lanes(jg, E, G, TG, k):
    """Groups that are no run of 1, 2, 4, 8 or 16 lanes are scored one at a time (equal scores among them)."""
    check_grouped(jg, 37, E, G, TG, k, 1.0)


@pytest.mark.parametrize("E,k", [(32, 2), (130, 8), (1000, 4)])
def test_nan_logits_leave_the_other_weights_alone(jg, E, k):
    """A NaN's key ranks above (sign bit clear) or below every number; its probability is exp_det's lower end and the
    others' are those of the numbers alone."""
    print("NaN logits", E, k, flush=True)
    rng = H.rng_for(E)
    logits = rng.standard_normal((9, E), dtype=np.float32)
    for t in range(8):
        logits[t, rng.integers(E)] = np.nan if t % 2 else -np.nan
    logits[7] = np.nan
    idx, w = (a.cpu().numpy() for a in jg.route_softmax_topk(H.to_cuda(logits), k))
    nan = np.isnan(logits)
    rank = np.where(nan, np.where(np.signbit(logits), -np.inf, np.inf), logits)
    assert np.array_equal(idx, np.argsort(-rank, axis=1, kind="stable")[:, :k])
    number = np.where(nan, np.float32(-np.inf), logits)
    number[7] = 0                                            # (no number at all: every expert the same)
    e = O.exp_det(number - number.max(axis=1, keepdims=True))
    p = np.take_along_axis(e / e.sum(axis=1, keepdims=True, dtype=np.float32), idx, axis=1)
    assert np.allclose(w, p / p.sum(axis=1, keepdims=True), rtol=2e-6, atol=1e-9)


@pytest.mark.parametrize("M,D", [(2, 2048), (2, 2176), (3, 4096), (1, 4224), (300, 1024)])
def test_rmsnorm_row_lengths(jg, M, D):
    check_rmsnorm(jg, M, D)


@pytest.mark.parametrize("M,offset", [(3, 0), (300, 0), (5, 1)])
def test_f32_activations_give_the_bits_of_their_bf16_rounding(jg, M, offset):
    """moe.py:282: the layer computes from bf16(x) and returns the caller's dtype, also for a view at an odd offset."""
    import torch
    print("f32 activations", M, offset, flush=True)
    D = 512
    params, _ = _layer(jg, D, 16, 256, 128, 9)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M)
    x = torch.randn(M * D + offset, device="cuda", generator=gen)[offset:].view(1, M, D)
    norm = torch.randn(D, device="cuda", generator=gen) * 0.1
    xb = x.to(torch.bfloat16)
    got, want = jg.moe_layer(x, params, 4), jg.moe_layer(xb, params, 4)
    assert got.dtype == torch.float32 and torch.equal(got, want.float())
    got, want = jg.moe_sublayer(x, norm, params, 4), jg.moe_sublayer(xb, norm, params, 4)
    assert got.dtype == torch.float32 and torch.equal(got, want.float())


@pytest.mark.parametrize("D,E,SI,dtype", [(512, 16, 128, "bf16"), (2176, 40, 0, "f32"), (4096, 130, 128, "bf16"), (4224, 8, 0, "bf16"),
                                          (8192, 1000, 128, "bf16")])   # (the last: K slices longer than a quantisation group)
def test_few_tokens_behind_the_norm_give_the_bits_of_a_larger_batch(jg, D, E, SI, dtype):
    """Up to four tokens take norm, quantiser and router matmul in one launch, five take two."""
    import torch
    print("norm and router", D, E, SI, dtype, flush=True)
    params, rand = _layer(jg, D, E, 128, SI, D)
    x = rand(1, 5, D).to(torch.float32 if dtype == "f32" else torch.bfloat16) * 3
    norm = rand(D).float() * 0.1
    x[0, 1] = 0                                              # an all-zero row
    want = jg.moe_sublayer(x, norm, params, 2)
    names = ("gate_proj", "up_proj", "down_proj")
    sorted_want, _ = jg.moe._forward(x[0], None, 2, params, shared={n: params["shared_" + n] for n in names} if SI else None,   # the grouped route
                                     gate_weight=params["gate_weight"], norm_weight=norm, add_residual=True, io_f32=dtype == "f32",
                                     shared_expert_gate_weight=params["shared_expert_gate_weight"] if SI else None, return_debug=True)
    assert torch.equal(sorted_want, want[0])
    for m in (1, 2, 3, 4):
        assert torch.equal(jg.moe_sublayer(x[:, :m].contiguous(), norm, params, 2), want[:, :m]), f"{m} tokens"


@pytest.mark.parametrize("M,E", [(1030, 24), (1030, 16)])   # 2060 rows: scales read row-major up to 96 rows an expert, gathered above
def test_scale_layouts_of_middle_sized_batches_give_the_same_bits(jg, M, E):
    import torch
    print("scale layouts", M, E, flush=True)
    params, rand = _layer(jg, 512, E, 256, 128, M + E)
    x, lg = rand(M, 512), rand(M, E).float()
    kw = dict(top_k=2, experts={n: params[n] for n in ("gate_proj", "up_proj", "down_proj")},
              shared={n: params["shared_" + n] for n in ("gate_proj", "up_proj", "down_proj")})
    whole = jg.moe_experts(x, lg, **kw)
    assert torch.equal(whole, jg.moe_experts(x, lg, return_debug=True, **kw)[0])      # (h scales row-major)
    assert torch.equal(whole[:400], jg.moe_experts(x[:400].contiguous(), lg[:400].contiguous(), **kw))


PLACED = [(1030, 128), (1030, 384), (4097, 640), (8192, 2048), (8193, 2048), (1100, 2176)]   # M, D; the last two: by a launch of its own


@pytest.mark.parametrize("M,D", PLACED)
def test_scales_that_the_sort_places_give_the_bits_of_rows_read_in_place(jg, M, D):
    """1, 3, 5, 16 and 17 scales a row, up to 2^18 of them and above, with dropped entries of a given selection and without."""
    import torch
    print("placed scales", M, D, flush=True)
    E = 12
    params, rand = _layer(jg, D, E, 128, 0, M + D)
    names = ("gate_proj", "up_proj", "down_proj")
    x, lg = rand(M, D), rand(M, E).float()
    kw = dict(top_k=2, experts={n: params[n] for n in names})
    whole, dbg = jg.moe_experts(x, lg, return_debug=True, **kw)
    assert torch.equal(jg.moe_experts(x, lg, **kw), whole)
    for lo in (0, M - 500):   # (1000 rows: scales read row-major)
        assert torch.equal(jg.moe_experts(x[lo:lo + 500].contiguous(), lg[lo:lo + 500].contiguous(), **kw), whole[lo:lo + 500])
    idx = dbg["indices"].clone()
    idx[::7, 0] = -1
    idx[3::11, 1] = E
    run = lambda rows: jg.expert_forward_single(x[rows].contiguous(), idx[rows].contiguous(), dbg["weights"][rows].contiguous(), *[params[n] for n in names])
    whole = run(slice(None))
    for lo in (0, M - 500):
        assert torch.equal(run(slice(lo, lo + 500)), whole[lo:lo + 500])


@pytest.mark.parametrize("R,D,I", [(4096, 256, 8192), (2090, 8192, 256), (5000, 512, 512)])   # (the last: lists of 53 and 79 tiles)
def test_one_group_of_many_rows_gives_the_bits_of_fewer(jg, R, D, I):
    """More than 768 work items of one group, whose height follows from the rounds that its rows make; and many short tiles."""
    import torch
    print("one group", R, D, I, flush=True)
    params, rand = _layer(jg, D, 1, I, 0, R)
    xq, sx = jg.quant_act(rand(R, D))
    run = lambda lo, hi: jg.gemm_gateup_swiglu(xq[lo:hi], sx[lo:hi].clone(), params["gate_proj"], params["up_proj"],
                                               H.to_cuda(np.array([0, hi - lo], np.int32)))
    hq, sh = run(0, R)
    y = jg.gemm_down(hq, sh, params["down_proj"], H.to_cuda(np.array([0, R], np.int32)))
    for lo, hi in ((0, 300), (700, 1300), (R - 33, R)):
        hq1, sh1 = run(lo, hi)
        assert torch.equal(hq1.view(torch.uint8), hq[lo:hi].view(torch.uint8)) and torch.equal(sh1, sh[lo:hi])
        assert torch.equal(jg.gemm_down(hq1, sh1, params["down_proj"], H.to_cuda(np.array([0, hi - lo], np.int32))), y[lo:hi])


@pytest.mark.parametrize("D,I,E,sizes", [
    (1024, 1024, 8, [512, 600, 700, 33, 520, 96, 1, 1634]),   # several tiles of 96 to 160 rows an expert
    (7168, 256, 4, [768, 384, 256, 192]),                     # 9 unequal tiles x 28 column blocks: one round, equal counts
    (512, 256, 32, [0, 200, 0, 1, 40] + [0] * 26 + [15]), (512, 256, 32, [0, 200, 0, 1, 40] + [0] * 26 + [16]),
    (512, 256, 1, [8]), (512, 256, 1, [9])])
def test_work_lists_of_few_and_more_rows_give_the_same_bits(jg, D, I, E, sizes):
    """8 rows an expert and one more: the two orders of the row-tile list (an expert of several tiles among empty ones).
    And a small problem whose experts are cut into several short tiles, for which weight lines are not marked as read once."""
    import torch
    print("work list", E, sum(sizes), flush=True)
    params, rand = _layer(jg, D, E, I, 0, E)
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    xq, sx = jg.quant_act(rand(int(off[-1]), D))
    hq, sh = jg.gemm_gateup_swiglu(xq, sx, params["gate_proj"], params["up_proj"], H.to_cuda(off))
    y = jg.gemm_down(hq, sh, params["down_proj"], H.to_cuda(off))
    for e in np.flatnonzero(sizes):
        lo, hi = int(off[e]), int(off[e + 1])
        one = {n: {k: v[e:e + 1] for k, v in params[n + "_proj"].items()} for n in ("gate", "up", "down")}
        o1 = H.to_cuda(np.array([0, hi - lo], np.int32))
        hq1, sh1 = jg.gemm_gateup_swiglu(xq[lo:hi], sx[lo:hi].clone(), one["gate"], one["up"], o1)
        assert torch.equal(hq1.view(torch.uint8), hq[lo:hi].view(torch.uint8)) and torch.equal(sh1, sh[lo:hi]), f"expert {e}: h"
        assert torch.equal(jg.gemm_down(hq1, sh1, one["down"], o1), y[lo:hi]), f"expert {e}: y"


SHORT = [33, 0, 1, 0, 2, 0, 0, 17, 0, 1, 0, 0, 16, 0, 3, 0, 0, 0, 32, 0, 0, 1, 0, 0, 0, 0, 0]   # at most 4 rows an expert on average
TALL = [250, 129, 128, 97, 96, 65, 64, 33, 1] + [0] * 47                                             # at most 16
MIXED = [129, 128, 97, 65, 33, 0, 1, 2, 2, 1, 0, 1] + [2] * 48 + [0] * 46                             # 574 rows in 64 tiles: two stages of the short ones


@pytest.mark.parametrize("E,D,I,sizes", [
    (108, 1024, 512, SHORT),      # 160 items of each GEMM: two stages
    (108, 1024, 1024, SHORT),     # 320 gate/up items: one stage
    (162, 256, 1536, SHORT),      # 720: more than all that run at once, two stages
    (162, 640, 512, SHORT),       # the last column block of the down GEMM is half full
    (108, 128, 512, SHORT),       # gate/up of one K step
    (405, 256, 128, SHORT),       # 150 items each, of two K steps and of one
    (405, 256, 256, SHORT),       # 300 gate/up items of two K steps, one stage
    (54, 2176, 1280, SHORT),      # weights from memory: copies of experts of one tile are non-temporal
    (56, 2048, 384, TALL),        # down tiles of up to 128 rows, plain copies ...
    (56, 2048, 1024, TALL),       # ... and non-temporal ones
    (106, 2048, 384, MIXED), (106, 2048, 1024, MIXED), (106, 1024, 128, MIXED),   # (the last: one K step)
])
def test_streamed_short_tiles_give_the_same_bits(jg, E, D, I, sizes):
    """Many short work items, which a kernel of their own takes: each expert's rows against a call of that expert alone
    (too few items for it), and one expert of every height against the oracle."""
    import torch
    print("streamed tiles", E, D, I, flush=True)
    sizes = [sizes[i % len(sizes)] for i in range(E)]
    params, rand = _layer(jg, D, E, I, 0, E + D)
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    R = int(off[-1])
    ids = H.to_cuda(H.rng_for(E + D + I).permutation(R).astype(np.int32))
    xq, sx = jg.quant_act(rand(R, D))
    hq, sh = jg.gemm_gateup_swiglu(xq, sx, params["gate_proj"], params["up_proj"], H.to_cuda(off), row_ids=ids)
    y = jg.gemm_down(hq, sh, params["down_proj"], H.to_cuda(off))
    gathered = jg.gather_scales(sx, ids)
    hb, sb = jg.gemm_gateup_swiglu(xq, gathered, params["gate_proj"], params["up_proj"], H.to_cuda(off), row_ids=ids, block_major=True)
    assert torch.equal(hb.view(torch.uint8), hq.view(torch.uint8)) and torch.equal(sb.t(), sh)
    assert torch.equal(jg.gemm_down(hb, sb, params["down_proj"], H.to_cuda(off), block_major=True), y)
    seen, got_h, want_h = set(), [], []
    for e in [e for e in range(min(E, 60)) if sizes[e]]:
        lo, hi = int(off[e]), int(off[e + 1])
        one = {n: {k: v[e:e + 1] for k, v in params[n + "_proj"].items()} for n in ("gate", "up", "down")}
        o1 = H.to_cuda(np.array([0, hi - lo], np.int32))
        hq1, sh1 = jg.gemm_gateup_swiglu(xq, sx, one["gate"], one["up"], o1, row_ids=ids[lo:hi].clone())
        assert torch.equal(hq1.view(torch.uint8), hq[lo:hi].view(torch.uint8)) and torch.equal(sh1, sh[lo:hi]), f"expert {e}: h"
        assert torch.equal(jg.gemm_down(hq1, sh1, one["down"], o1), y[lo:hi]), f"expert {e}: y"
        if sizes[e] not in seen:                                 # one expert of every height: both GEMMs against the oracle
            seen.add(sizes[e])
            rows, o1 = ids[lo:hi].long(), np.array([0, hi - lo], np.int32)
            experts = {n: (H.codes_np(one[n]["w"]), one[n]["scale_inv"].cpu().numpy()) for n in one}
            xe = H.codes_np(xq[rows]), sx[rows].cpu().numpy()
            got_h.append((H.codes_np(hq[lo:hi]), sh[lo:hi].cpu().numpy()))
            want_h.append(O.expert_swiglu(*xe, experts, o1)[1:])
            want = O.grouped_gemm(H.codes_np(hq[lo:hi]), sh[lo:hi].cpu().numpy(), *experts["down"], o1)
            H.assert_close_out(H.bf16_to_np(y[lo:hi]), O.bf16_round(want.astype(np.float32)))
    # (all of them together, 11000 codes at least: one row of 512 codes has some one that lie on a rounding boundary, and more
    # than the helper's two in one row of twelve -- Poisson at the 0.2 % that it tells of)
    H.assert_h_close(*map(np.concatenate, zip(*got_h)), *map(np.concatenate, zip(*want_h)), "h of the sampled experts")


@pytest.mark.parametrize("routing", ["softmax", "sigmoid_grouped"])
def test_batches_of_every_tile_height_give_the_bits_of_a_large_one(jg, routing):
    """5 to 600 tokens of one layer with a shared expert: tiles of 32 and 128 rows in the two GEMMs' kernels."""
    import torch
    print("batches", routing, flush=True)
    D, E, I, SI, k = 1152, 128, 512, 256, 4
    params, rand = _layer(jg, D, E, I, SI, 11)
    M = 4000
    x, lg = rand(M, D), rand(M, E).float()
    kw = dict(top_k=k, experts={n: params[n] for n in ("gate_proj", "up_proj", "down_proj")}, routing=routing,
              shared={n: params["shared_" + n] for n in ("gate_proj", "up_proj", "down_proj")})
    if routing == "sigmoid_grouped":
        kw.update(n_group=8, topk_group=4, bias=0.1 * torch.arange(E, device="cuda").remainder(5).float())
    whole = jg.moe_experts(x, lg, **kw)
    for m in (5, 32, 33, 128, 129, 600):
        assert torch.equal(jg.moe_experts(x[:m].contiguous(), lg[:m].contiguous(), **kw), whole[:m]), f"{m} tokens"


@pytest.mark.parametrize("M,E,k", [(1793, 40, 2), (2047, 8, 1), (4099, 128, 8)])
def test_many_tokens_a_workgroup_are_routed_exactly(jg, M, E, k):
    """8 to 17 tokens of a routing workgroup, of eight waves beside the quantiser; the last one has fewer."""
    test_ready_logits_routed_and_sorted_in_one_launch_or_two(jg, M, E, k)


@pytest.mark.parametrize("n,KB", [(1, 1), (257, 3), (300, 4), (255, 16), (70, 17), (513, 20), (256, 56), (5, 64 * 16 + 8), (5, 64 * 16 + 9)])
def test_scales_are_gathered_whole(jg, n, KB):
    """Rows of fewer and more scales than a thread takes and than the grid covers at once, a multiple of four or not."""
    import torch
    print("scales", n, KB, flush=True)
    sx = torch.arange(2 * n * KB, dtype=torch.float32, device="cuda").reshape(2 * n, KB)
    ids = torch.randperm(2 * n, device="cuda")[:n].to(torch.int32)
    assert torch.equal(jg.gather_scales(sx, ids), sx[ids.long()].t())
    assert torch.equal(jg.gather_scales(sx, n_rows=n), sx[:n].t())


@pytest.mark.parametrize("R", [2100, 2600, 6100, 9000])   # (the first: 32 tiles of 16 column blocks, two full rounds: no large pool)
def test_uneven_groups_that_are_drawn_give_the_same_bits(jg, R):
    """Few rounds of long items of uneven groups: most of the list is a pool that the XCDs draw from (empty experts, one of
    many tiles and of one row among them).  And the even split of the same rows, whose pool is small."""
    import torch
    E, D, I = 32, 1536, 2048
    print("uneven groups", R, flush=True)
    params, rand = _layer(jg, D, E, I, 0, R)
    p = 1.0 / np.arange(1, E + 1) ** 1.2
    p[[5, 17, 30]] = 0.0
    uneven = np.floor(p / p.sum() * (R - 40)).astype(np.int64)
    uneven[31] = 1
    uneven[0] += R - uneven.sum()
    xq, sx = jg.quant_act(rand(R, D))
    for sizes in (uneven, np.full(E, R // E) + (np.arange(E) < R % E)):
        off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
        hq, sh = jg.gemm_gateup_swiglu(xq, sx, params["gate_proj"], params["up_proj"], H.to_cuda(off))
        y = jg.gemm_down(hq, sh, params["down_proj"], H.to_cuda(off))
        for e in np.flatnonzero(sizes):
            lo, hi = int(off[e]), int(off[e + 1])
            one = {n: {k: v[e:e + 1] for k, v in params[n + "_proj"].items()} for n in ("gate", "up", "down")}
            o1 = H.to_cuda(np.array([0, hi - lo], np.int32))
            hq1, sh1 = jg.gemm_gateup_swiglu(xq[lo:hi], sx[lo:hi].clone(), one["gate"], one["up"], o1)
            assert torch.equal(hq1.view(torch.uint8), hq[lo:hi].view(torch.uint8)) and torch.equal(sh1, sh[lo:hi]), f"expert {e}: h"
            assert torch.equal(jg.gemm_down(hq1, sh1, one["down"], o1), y[lo:hi]), f"expert {e}: y"


@pytest.mark.parametrize("D,E,I,k,M,spread", [
    (1664, 16, 2048, 3, 1500, 1.5),
    (4096, 32, 640, 2, 250, 20.0),   # tiles of up to 128 rows, weights from memory
])
def test_uneven_routing_of_a_layer_of_few_experts(jg, D, E, I, k, M, spread):
    """The same list inside the layer, written by the sort and read by both GEMMs: the output against its own stages."""
    import torch
    print("uneven layer", D, E, flush=True)
    params, rand = _layer(jg, D, E, I, 0, 9)
    x, lg = rand(M, D), rand(M, E).float() + spread * torch.linspace(1, 0, E, device="cuda")
    ex = {n: params[n] for n in ("gate_proj", "up_proj", "down_proj")}
    out, dbg = jg.moe_experts(x, lg, top_k=k, experts=ex, return_debug=True)
    assert torch.equal(out, jg.moe_experts(x, lg, top_k=k, experts=ex))
    assert int(dbg["group_sizes"].max()) > max(2 * M * k // E, 128)
    off = torch.cat([torch.zeros(1, dtype=torch.int32, device="cuda"), dbg["group_sizes"].cumsum(0).to(torch.int32)])
    xq, sx = jg.quant_act(x)
    for e in [e for e in range(E) if off[e + 1] > off[e]]:
        lo, hi = int(off[e]), int(off[e + 1])
        one = {n: {k2: v[e:e + 1] for k2, v in ex[n].items()} for n in ex}
        o1 = H.to_cuda(np.array([0, hi - lo], np.int32))
        hq1, sh1 = jg.gemm_gateup_swiglu(xq, sx, one["gate_proj"], one["up_proj"], o1, row_ids=dbg["sorted_token_ids"][lo:hi].clone())
        assert torch.equal(hq1.view(torch.uint8), dbg["hq"][lo:hi]), f"expert {e}: h"
        assert torch.equal(jg.gemm_down(hq1, sh1, one["down_proj"], o1), dbg["y"][lo:hi]), f"expert {e}: y"


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_activations_in_any_strides(jg, dtype):
    """The layer takes (B, T, D) activations as they lie; the flat entry points take two dimensions and refuse others."""
    import torch
    print("strides", dtype, flush=True)
    params, rand = _layer(jg, 256, 8, 128, 128, 5)
    x = rand(3, 5, 256).to(getattr(torch, dtype))
    want = jg.moe_layer(x, params, 2)
    assert want.shape == x.shape and want.dtype == x.dtype and want.is_contiguous()
    for other in (x.transpose(0, 1).contiguous().transpose(0, 1), torch.cat([x, x], 2)[..., :256]):
        assert not other.is_contiguous()
        got = jg.moe_layer(other, params, 2)
        assert torch.equal(got, want) and got.is_contiguous()
    for bad in (x[0, 0], x[None]):
        with pytest.raises(ValueError):
            jg.moe_layer(bad, params, 2)
    ex = {n: params[n] for n in ("gate_proj", "up_proj", "down_proj")}
    for bad in (x.to(torch.bfloat16), x[0, 0].to(torch.bfloat16)):
        with pytest.raises(ValueError):
            jg.moe_experts(bad, rand(15, 8).float(), top_k=2, experts=ex)


@pytest.mark.parametrize("M,k,E", [(1, 1, 1), (1, 8, 256), (4, 8, 64), (31, 1, 65), (32, 1, 1), (1, 32, 1024), (3, 11, 130), (5, 7, 8)])
def test_few_entries_are_sorted(jg, M, k, E):
    """Up to 32 entries and one more, any number of one expert among them."""
    import torch
    print("few entries", M, k, E, flush=True)
    rng = H.rng_for(M * 100 + k + E)
    for idx in (rng.integers(0, E, (M, k)), np.full((M, k), E - 1), np.arange(M * k).reshape(M, k)[::-1] % E):
        idx = np.ascontiguousarray(idx.astype(np.int32))
        got, ref = jg.permute(H.to_cuda(idx), E), O.sort_and_group(idx, E)
        for name in ("group_sizes", "group_offsets", "sorted_token_ids", "sort_order", "inv_perm"):
            if name in ref:
                assert np.array_equal(got[name].cpu().numpy(), ref[name]), name


@pytest.mark.parametrize("M,k,E", [(4, 8, 24), (8, 4, 24), (16, 2, 8), (11, 3, 24)])
def test_few_entries_of_a_layer(jg, M, k, E):
    """The same inside the layer, routed (up to 32 entries are sorted by the routing launch) or given, all rows of one expert too."""
    import torch
    print("few entries of a layer", M, k, E, flush=True)
    params, rand = _layer(jg, 256, E, 256, 0, M)
    ex = [params[n] for n in ("gate_proj", "up_proj", "down_proj")]
    x, lg = rand(200, 256), rand(200, E).float()
    kw = dict(top_k=k, experts=dict(zip(("gate_proj", "up_proj", "down_proj"), ex)))
    whole = jg.moe_experts(x, lg, **kw)
    assert torch.equal(jg.moe_experts(x[:M].contiguous(), lg[:M].contiguous(), **kw), whole[:M])
    got, dbg = jg.moe_experts(x[:M].contiguous(), lg[:M].contiguous(), return_debug=True, **kw)   # (sorted, not straight to the experts)
    ref = O.sort_and_group(dbg["indices"].cpu().numpy(), E)
    assert torch.equal(got, whole[:M])
    for name in ("group_sizes", "sorted_token_ids", "inv_perm"):
        assert np.array_equal(dbg[name].cpu().numpy(), ref[name]), name
    w = rand(M, k).float()
    same = torch.full((M, k), E - 2, dtype=torch.int32, device="cuda")
    many = same.repeat(20, 1)
    got = jg.expert_forward_single(x[:M].contiguous(), same, w, *ex)
    assert torch.equal(got, jg.expert_forward_single(x[:M].repeat(20, 1), many, w.repeat(20, 1), *ex)[:M])


@pytest.mark.parametrize("M,D,E,k,I,SI", [
    (1, 128, 8, 2, 128, 0),       # one K step, eight tiles
    (16, 512, 8, 2, 1024, 0),     # the most tokens, two tiles a workgroup
    (9, 1024, 8, 2, 256, 0),      # three: some span two scale blocks, and the last workgroup has one
    (13, 384, 33, 3, 256, 384),   # a shared expert wider than the routed ones
    (3, 896, 40, 17, 128, 128),   # more slots than waves
    (2, 256, 40, 32, 256, 128),   # the most slots
    (16, 4096, 4, 1, 128, 128),   # sixteen tiles a workgroup
    (1, 2048, 8, 8, 2432, 128),   # longer rows of the routed experts than of the shared one
    (1, 128, 8, 8, 13312, 128),   # rows whose rings do not fit beside each other for every slot
    (1, 7168, 18, 8, 512, 512),   # one token of a layer from memory (non-temporal copies) ...
    (2, 7168, 18, 8, 512, 512),   # ... and two
])
@pytest.mark.parametrize("f32", [False, True])
def test_experts_of_single_tokens_give_the_grouped_bits(jg, M, D, E, k, I, SI, f32):
    """Batches that go from the selection straight to the experts: the bits of the grouped kernels (the call that returns
    the sorted intermediates), routed or given, with norm, gate and residual, also where h or the rows hold infinities and NaN."""
    import torch
    print("single tokens", M, D, E, k, I, SI, f32, flush=True)
    same = lambda a, b: torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(7.0, float("inf"), -float("inf")), b.nan_to_num(7.0, float("inf"), -float("inf")))
    params, rand = _layer(jg, D, E, I, SI, M + D)
    names = ("gate_proj", "up_proj", "down_proj")
    ex = {n: params[n] for n in names}
    x = rand(M, D)
    for hard in (False, True):
        if hard:
            x[0, 5], x[M - 1, D - 1] = 3e38, -3e38
            if M > 2:
                x[1, 0], x[2, 1] = float("inf"), float("nan")
        kw = dict(top_k=k, experts=ex, gate_weight=params["gate_weight"])
        if SI:
            kw.update(shared={n: params["shared_" + n] for n in names}, norm_weight=torch.rand(D, device="cuda") + 0.5,
                      shared_expert_gate_weight=params["shared_expert_gate_weight"], add_residual=True)
        if f32:
            fwd = lambda **o: jg.moe._forward(x.float(), None, io_f32=True, **kw, **o)
        else:
            fwd = lambda **o: jg.moe_experts(x, None, **kw, **o)
        want, dbg = fwd(return_debug=True)
        assert same(fwd(), want)
        if not SI:
            given = [params[n] for n in names]
            got = jg.expert_forward_single(x, dbg["indices"], dbg["weights"], *given)
            assert same(got, want.to(got.dtype))
            w = dbg["weights"].clone()                           # infinite rows of the output, by a weight; the same tokens
            w[M - 1, 0] = float("inf")                           # often enough to be grouped
            got = jg.expert_forward_single(x, dbg["indices"], w, *given)
            many = jg.expert_forward_single(x.repeat(20, 1), dbg["indices"].repeat(20, 1), w.repeat(20, 1), *given)
            assert same(got, many[:M]) and (hard or got[M - 1].isinf().any())
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        out = fwd()
    for i in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert same(out, want), f"replay {i}"


ROUTED_TOKENS = [   # M, D, E, k, I, SI of ready logits: routed by the experts' first launch, or just not
    (1, 128, 1, 1, 128, 0), (3, 384, 128, 3, 256, 128), (3, 4096, 129, 4, 128, 0), (1, 4224, 256, 8, 256, 128), (1, 7168, 64, 8, 2048, 256),
    (1, 512, 257, 2, 256, 0), (16, 512, 8, 2, 1024, 0), (16, 1024, 64, 8, 384, 0), (1, 7168, 32, 8, 3072, 0)]


@pytest.mark.parametrize("routing", ["softmax", "sigmoid_grouped"])
@pytest.mark.parametrize("M,D,E,k,I,SI", ROUTED_TOKENS)
def test_ready_logits_of_single_tokens_give_the_grouped_bits(jg, M, D, E, k, I, SI, routing):
    """Routing and quantiser inside the experts' first launch: the bits of the call that launches them one by one, also with logits
    that are equal, infinite or NaN and rows that are zero or hold infinities and NaN; other rows in replays of a graph."""
    import torch
    print("ready logits of single tokens", M, D, E, k, I, SI, routing, flush=True)
    params, rand = _layer(jg, D, E, I, SI, M + D + E)
    names = ("gate_proj", "up_proj", "down_proj")
    kw = dict(top_k=k, experts={n: params[n] for n in names}, routing=routing, shared={n: params["shared_" + n] for n in names} if SI else None)
    if routing == "sigmoid_grouped":
        groups = 8 if E % 8 == 0 else 1
        kw.update(bias=0.1 * torch.arange(E, device="cuda").remainder(5).float(), routed_scale=2.5, n_group=groups, topk_group=max(groups // 2, 1))
        if k > kw["topk_group"] * (E // groups):
            kw.update(n_group=1, topk_group=1)
    same = lambda a, b: torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(7.0, float("inf"), -float("inf")), b.nan_to_num(7.0, float("inf"), -float("inf")))
    rows = []
    for kind in ("plain", "ties", "odd logits", "zero rows", "odd rows"):
        x, lg = rand(M, D), rand(M, E).float()
        if kind == "ties":
            lg = lg.round()
        if kind == "odd logits":
            lg[0, 0], lg[M - 1, E // 2], lg[0, E - 1] = float("nan"), float("inf"), -float("inf")
        if kind == "zero rows":
            x[M - 1] = 0
        if kind == "odd rows":
            x[0, 5], x[M - 1, D - 1] = float("inf"), float("nan")
        want, dbg = jg.moe_experts(x, lg, return_debug=True, **kw)
        assert same(jg.moe_experts(x, lg, **kw), want), kind
        if not SI:
            given = jg.expert_forward_single(x, dbg["indices"], dbg["weights"], *[params[n] for n in names])
            assert same(given, want.to(given.dtype)), kind
        rows.append((x, lg, want))
    x, lg = rows[0][0].clone(), rows[0][1].clone()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        out = jg.moe_experts(x, lg, **kw)
    for i, (xi, li, want) in enumerate(rows):
        x.copy_(xi), lg.copy_(li), out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert same(out, want), f"replay {i}"


FRONTED_TOKENS = [   # M, D, E, k, I, SI, norm: behind a small router, in the experts' first launch, or just not
    (1, 1024, 32, 2, 512, 512, True), (3, 1024, 32, 2, 512, 512, True), (5, 1024, 32, 2, 512, 512, False), (4, 1024, 32, 2, 512, 512, True),
    (2, 640, 64, 4, 128, 256, True), (1, 512, 64, 8, 256, 0, False), (2, 128, 1, 1, 128, 128, True), (16, 256, 16, 2, 256, 0, False), (1, 896, 17, 3, 384, 128, True)]


@pytest.mark.parametrize("routing", ["softmax", "sigmoid_grouped"])
@pytest.mark.parametrize("M,D,E,k,I,SI,norm", FRONTED_TOKENS)
def test_small_routers_of_single_tokens_give_the_grouped_bits(jg, M, D, E, k, I, SI, norm, routing):
    """Norm, router and selection inside the experts' first launch: the bits of the call that takes them launch by launch."""
    import torch
    print("small routers of single tokens", M, D, E, k, I, SI, norm, routing, flush=True)
    params, rand = _layer(jg, D, E, I, SI, M + D + E)
    names = ("gate_proj", "up_proj", "down_proj")
    same = lambda a, b: torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(7.0, float("inf"), -float("inf")), b.nan_to_num(7.0, float("inf"), -float("inf")))
    kw = dict(top_k=k, experts={n: params[n] for n in names}, routing=routing, gate_weight=params["gate_weight"], add_residual=True)
    if SI:
        kw.update(shared={n: params["shared_" + n] for n in names}, shared_expert_gate_weight=params["shared_expert_gate_weight"])
    if norm:
        kw.update(norm_weight=rand(D).float() * 0.1)
    if routing == "sigmoid_grouped":
        kw.update(bias=0.1 * torch.arange(E, device="cuda").remainder(5).float())
    for kind in ("plain", "zero rows", "odd rows"):
        x = rand(M, D)
        if kind == "zero rows":
            x[M - 1] = 0
        if kind == "odd rows":
            x[0, 5], x[M - 1, D - 1] = float("inf"), float("nan")
        for f32 in (False, True):
            run = lambda **o: jg.moe._forward(x.float() if f32 else x, None, io_f32=f32, **kw, **o)
            assert same(run(), run(return_debug=True)[0]), (kind, f32)


@pytest.mark.parametrize("M,k", [(1, 2), (5, 3), (16, 8),     # straight to the experts, read by their first launch, which quantises too
                                 (17, 1), (32, 1), (17, 3),   # the sort without counters, and with them
                                 (700, 2), (1100, 2), (3000, 3)])   # scales read row-major, and gathered; several chunks
def test_selected_experts_that_there_are_not_count_as_zero_rows(jg, M, k):
    """A given selection may hold indices outside [0, E): their entries are dropped by the sort and add nothing."""
    import torch
    print("dropped entries", M, k, flush=True)
    D, E, I = 512, 10, 256
    params, rand = _layer(jg, D, E, I, 0, M + k)
    ex = [params[n] for n in ("gate_proj", "up_proj", "down_proj")]
    rng = H.rng_for(M * 10 + k)
    idx = rng.integers(0, E, (M, k))
    drop = rng.random((M, k)) < 0.3
    drop[0] = True                                            # a token with no expert at all
    bad = np.where(drop, rng.choice([-1, E, 2 ** 31 - 1, -2 ** 31], (M, k)), idx).astype(np.int32)
    w = np.abs(rng.standard_normal((M, k))).astype(np.float32)
    x = rand(M, D)
    got = jg.expert_forward_single(x, H.to_cuda(bad), H.to_cuda(w), *ex)
    want = jg.expert_forward_single(x, H.to_cuda(idx.astype(np.int32)), H.to_cuda(np.where(drop, np.float32(0), w)), *ex)
    assert torch.equal(got, want) and not got[0].any()
    p = jg.permute(H.to_cuda(bad), E)
    n, flat = int((~drop).sum()), np.flatnonzero(~drop.reshape(-1))
    order = flat[np.argsort(bad.reshape(-1)[flat], kind="stable")]
    inv = np.full(M * k, -1)
    inv[order] = np.arange(n)
    assert np.array_equal(p["sort_order"].cpu().numpy()[:n], order) and np.array_equal(p["sorted_token_ids"].cpu().numpy()[:n], order // k)
    assert not p["sort_order"][n:].any() and not p["sorted_token_ids"][n:].any()   # (a walk to the lists' ends stays inside the rows)
    _, sx = jg.quant_act(x)
    assert torch.equal(jg.gather_scales(sx, p["sorted_token_ids"]), sx[p["sorted_token_ids"].long()].t())
    assert np.array_equal(p["inv_perm"].cpu().numpy(), inv) and int(p["group_offsets"][-1]) == n
    assert np.array_equal(p["group_sizes"].cpu().numpy(), np.bincount(bad.reshape(-1)[flat], minlength=E))


DROPPED = (16, 512, 128, 8, 1024, 0)   # more workgroups than run at once: the first launch finds the tokens quantised


def test_selected_experts_that_there_are_not_leave_their_workgroups(jg):
    """The same of the first launch behind a quantiser of its own: workgroups without an expert end with copies under way."""
    import torch
    print("dropped entries of many workgroups", flush=True)
    M, D, E, k, I, _ = DROPPED
    params, rand = _layer(jg, D, E, I, 0, 5)
    ex = [params[n] for n in ("gate_proj", "up_proj", "down_proj")]
    rng = H.rng_for(11)
    idx = rng.integers(0, E, (M, k)).astype(np.int32)
    drop = rng.random((M, k)) < 0.4
    drop[3] = True
    w, x = np.abs(rng.standard_normal((M, k))).astype(np.float32), rand(M, D)
    bad = np.where(drop, rng.choice([-1, E, 2 ** 31 - 1, -2 ** 31], (M, k)), idx).astype(np.int32)
    for _ in range(3):
        got = jg.expert_forward_single(x, H.to_cuda(bad), H.to_cuda(w), *ex)
        want = jg.expert_forward_single(x, H.to_cuda(idx), H.to_cuda(np.where(drop, np.float32(0), w)), *ex)
        assert torch.equal(got, want) and not got[3].any()
    many = jg.expert_forward_single(x.repeat(20, 1), H.to_cuda(bad).repeat(20, 1), H.to_cuda(w).repeat(20, 1), *ex)   # (sorted)
    assert torch.equal(got, many[:M])


@pytest.mark.parametrize("E", [256, 257, 512, 640])
@pytest.mark.parametrize("M,D", [(1, 4096), (3, 2304), (256, 1152), (257, 2176)])
def test_partial_sums_of_wide_routers(jg, M, D, E):
    """Routing that adds the router's partial sums itself (9, 17, 18 and 32 slices; a thread a column up to 256 tokens)
    selects what the router's own logits select."""
    import torch
    print("wide routers", M, D, E, flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + E)
    x = torch.randn((M, D), dtype=torch.bfloat16, device="cuda", generator=gen)
    gate = torch.randn((E, D), dtype=torch.bfloat16, device="cuda", generator=gen).mul_(0.02).t()
    idx, w = jg.moe_routing(x, gate, 7)
    want_idx, want_w = jg.route_softmax_topk(jg.router_logits(x, gate), 7)
    assert torch.equal(idx.reshape(M, 7), want_idx) and torch.equal(w.reshape(M, 7), want_w.to(w.dtype))


TALL = dict(E=96, D=2048, I=1024)   # 8 column blocks and 16 or 8 K steps


@pytest.mark.parametrize("sizes", [
    [320, 289, 288, 200, 224, 225, 256, 240],     # one tile an expert, of 320 rows at most
    [320, 289, 1, 319, 313, 304, 290, 270],       # ... and of all heights from 33 rows up to there
    [320, 289, 0, 319, 313, 304, 290, 270],       # ... and none
    [321, 289, 288, 200, 224, 225, 256, 240],     # one row too many: full tiles
    [288, 287, 288, 224, 224, 225, 256, 240],     # ... no row too many
    [640, 577, 576, 480, 449, 512, 500, 511],     # two tiles an expert
])
def test_tall_tiles_give_the_bits_of_full_ones(jg, sizes):
    """Lists that may have tiles of 320 rows (what the host says of these batches: test_dispatch_rules.py) against the stage
    functions, whose lists have none."""
    import torch
    print("tall tiles", sizes, flush=True)
    E, D, I = TALL["E"], TALL["D"], TALL["I"]
    rows = np.array([sizes[i % len(sizes)] for i in range(E)])
    rng = np.random.default_rng(int(rows.sum()))
    idx = rng.permutation(np.repeat(np.arange(E), rows)).astype(np.int32)[:, None]
    M = len(idx)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M)
    rand = lambda *s: torch.randn(s, dtype=torch.bfloat16, device="cuda", generator=gen)
    ex = {n: jg.quantize_weight_block(rand(E, *s).mul_(0.02)) for n, s in (("gate_proj", (I, D)), ("up_proj", (I, D)), ("down_proj", (D, I)))}
    x, w, didx = rand(M, D), torch.rand(M, 1, device="cuda", generator=gen), H.to_cuda(idx)
    got = [jg.expert_forward_single(x, didx, w, *ex.values()) for _ in range(2)]
    p = jg.permute(didx, E)
    xq, sx = jg.quant_act(x)
    hq, sh = jg.gemm_gateup_swiglu(xq, sx, ex["gate_proj"], ex["up_proj"], p["group_offsets"], row_ids=p["sorted_token_ids"])
    want = jg.combine(jg.gemm_down(hq, sh, ex["down_proj"], p["group_offsets"]), w, p["inv_perm"])
    assert torch.equal(got[0], want) and torch.equal(got[1], want)


@pytest.mark.parametrize("M,D,E,SI,dtype,routing", [
    (1, 1024, 64, 128, "bf16", "softmax"),        # the widest router: 65 columns
    (3, 128, 1, 0, "f32", "softmax"),             # one K block, one expert
    (17, 384, 33, 128, "f32", "softmax"),         # half a wave of pieces a row, two columns beyond two fragments
    (256, 640, 16, 0, "bf16", "sigmoid_grouped"), # a wave and a quarter of pieces
    (257, 1024, 8, 128, "bf16", "softmax"),       # two tokens a workgroup, the last one alone
    (1025, 512, 40, 0, "bf16", "sigmoid_grouped"),   # eight, and selections counted for the sort
    (2049, 896, 12, 128, "f32", "softmax"),       # sixteen, block-major scales
    (4097, 256, 64, 0, "bf16", "softmax"),        # more workgroups than histograms (with the norm: launch by launch)
])
def test_small_routers_in_one_launch_give_the_bits_of_the_stages(jg, M, D, E, SI, dtype, routing):
    import torch
    print("one launch up to the selection", M, D, E, SI, dtype, routing, flush=True)
    params, rand = _layer(jg, D, E, 128, SI, M + D)
    names = ("gate_proj", "up_proj", "down_proj")
    k = min(2, E)
    kw = dict(routing=routing, n_group=4, topk_group=2, bias=rand(E).float() * 0.1, routed_scale=1.5) if routing != "softmax" else {}
    experts, shared = {n: params[n] for n in names}, {n: params["shared_" + n] for n in names} if SI else None
    x = rand(M, D).to(torch.float32 if dtype == "f32" else torch.bfloat16) * 3
    x[M // 2] = 0                                            # an all-zero row
    norm = rand(D).float() * 0.1
    odd = torch.empty(D + 1, device="cuda")[1:]              # (read 16 bytes at a time: this one goes launch by launch)
    odd.copy_(norm)
    run = lambda norm, **o: jg.moe._forward(x, None, k, experts, shared=shared, gate_weight=params["gate_weight"], norm_weight=norm, io_f32=dtype == "f32",
                                            shared_expert_gate_weight=params["shared_expert_gate_weight"] if SI else None, **kw, **o)
    # with the norm: against the same call launch by launch
    got, dbg = run(norm, add_residual=True, return_debug=True)
    want, ref = run(odd, add_residual=True, return_debug=True)
    for n in ref:
        assert torch.equal(dbg[n], ref[n]), n
    assert torch.equal(got, want) and torch.equal(run(norm, add_residual=True), want)
    # without: against the stages
    xb = x.bfloat16()
    stage = jg.router_logits(xb, params["gate_weight"], params["shared_expert_gate_weight"] if SI else None)
    logits, gate = stage if SI else (stage, None)
    got, dbg = run(None, return_debug=True)
    assert torch.equal(dbg["logits"], logits) and (not SI or torch.equal(dbg["shared_gate"], gate))
    idx, w = jg.route_softmax_topk(logits, k) if routing == "softmax" else jg.route_sigmoid_grouped(logits, kw["bias"], 4, 2, k, True, 1.5)
    assert torch.equal(dbg["indices"], idx) and torch.equal(dbg["weights"], w)
    assert torch.equal(got, run(None))
    if not SI:
        assert torch.equal(got.bfloat16(), jg.expert_forward_single(xb, idx, w, *experts.values()))
    if routing == "softmax":
        assert all(map(torch.equal, jg.moe_routing(xb, params["gate_weight"], k), (idx, w)))


SCANNED = [   # M, D, E, k, I, SI, offsets on the logits
    (17, 128, 1, 1, 128, 0, 0),       # one expert, one K step
    (33, 384, 8, 2, 256, 0, 0),       # a half-full last column block
    (64, 512, 64, 1, 128, 128, 0),    # as many experts as lanes; a shared expert beside
    (100, 640, 7, 3, 384, 0, 30),     # a few experts take all: several tiles each, experts without rows
    (512, 512, 8, 2, 1024, 0, 1),     # two selections a thread
    (1024, 256, 60, 2, 128, 0, 0),    # four: all that they hold
    (385, 256, 8, 4, 128, 128, 1),    # the last of four in a few waves
    (511, 1024, 32, 2, 512, 512, 2),  # uneven, with a shared expert in several tiles
    (128, 256, 33, 8, 256, 128, 0),   # eight selections a token
]


@pytest.mark.parametrize("M,D,E,k,I,SI,offset", SCANNED)
def test_small_layers_without_a_list_give_the_bits_of_the_sorted_rows(jg, M, D, E, k, I, SI, offset):
    """Where the GEMMs read the selection themselves (test_dispatch_rules.py says that these batches do) against the call whose
    sorted rows are asked for, which has a list."""
    import torch
    print("selection read by the GEMMs", M, D, E, k, I, SI, offset, flush=True)
    params, rand = _layer(jg, D, E, I, SI, M + D)
    names = ("gate_proj", "up_proj", "down_proj")
    experts = {n: params[n] for n in names}
    kw = dict(top_k=k, experts=experts, shared={n: params["shared_" + n] for n in names} if SI else None)
    x, lg = rand(M, D), rand(M, E).float() + offset * rand(E).float()
    want, dbg = jg.moe_experts(x, lg, return_debug=True, **kw)
    for _ in range(2):
        assert torch.equal(jg.moe_experts(x, lg, **kw), want)
    if SI:
        return
    assert torch.equal(jg.expert_forward_single(x, dbg["indices"], dbg["weights"], *experts.values()), want)
    # selections outside [0, E) have no row
    idx = dbg["indices"].clone()
    idx[::3, 0] = E
    idx[1::4, -1] = -7
    idx[2] = 1 << 30
    keep = (idx >= 0) & (idx < E)
    got = jg.expert_forward_single(x, idx, dbg["weights"], *experts.values())
    same = jg.expert_forward_single(x, torch.where(keep, idx, 0), torch.where(keep, dbg["weights"], 0.0), *experts.values())
    assert torch.equal(got, same) and not got[2].any()


TWO_LISTS = [   # M, D, E, k, I, SI, offset
    (1300, 1536, 128, 2, 768, 0, 0),      # 20 rows an expert: a tile each in both lists
    (3000, 1536, 128, 8, 768, 256, 0),    # about 188: one of gate/up, two of down; a shared expert beside
    (2100, 1792, 128, 6, 768, 0, 2),      # uneven: experts without rows and of several tiles of each kind; a half last column block
    (2000, 256, 800, 8, 768, 0, 0.5),     # more experts than the routing launch counts for
    (1500, 2048, 100, 4, 1024, 0, 0),     # as many K steps as there may be
]


@pytest.mark.parametrize("M,D,E,k,I,SI,offset", TWO_LISTS)
def test_a_down_gemm_with_its_own_list_gives_the_bits_of_small_batches(jg, M, D, E, k, I, SI, offset):
    """The same tokens in batches that one workgroup sorts, which have one list; and the rows of h and y that the two GEMMs share."""
    import torch
    print("two work lists", M, D, E, k, I, SI, offset, flush=True)
    params, rand = _layer(jg, D, E, I, SI, M)
    names = ("gate_proj", "up_proj", "down_proj")
    kw = dict(top_k=k, experts={n: params[n] for n in names}, shared={n: params["shared_" + n] for n in names} if SI else None)
    x, lg = rand(M, D), rand(M, E).float() + offset * rand(E).float()
    got = jg.moe_experts(x, lg, **kw)
    part = 2048 // k
    for t in range(0, M, part):
        want = jg.moe_experts(x[t:t + part].contiguous(), lg[t:t + part].contiguous(), **kw)
        assert torch.equal(got[t:t + part], want), t
    again, dbg = jg.moe_experts(x, lg, return_debug=True, **kw)
    assert torch.equal(again, got)
    idx = dbg["indices"].clone()
    idx[::5, 1] = E   # no expert: the lists are shorter than the batch
    w = torch.where(idx < E, dbg["weights"], 0.0)
    if not SI:
        full = jg.expert_forward_single(x, idx, w, *(params[n] for n in names))
        for t in range(0, M, part):
            assert torch.equal(full[t:t + part], jg.expert_forward_single(x[t:t + part].contiguous(), idx[t:t + part].contiguous(), w[t:t + part].contiguous(),
                                                                          *(params[n] for n in names))), t


SMALL_DOWN = [   # M, D, E, k, I, SI, selections a lane
    (17, 128, 1, 1, 128, 0, 1),        # one expert: units of 16 rows and of one
    (64, 256, 64, 1, 128, 128, 1),     # a workgroup's 64 selections, and a unit for nearly each; four of the shared expert
    (65, 128, 5, 1, 128, 0, 1),        # one more than a workgroup has
    (43, 384, 7, 3, 384, 256, 1),      # 63 selections of 21 tokens; an odd number of K steps
    (40, 256, 6, 20, 256, 0, 1),       # more of a token than there are experts, three tokens
    (200, 512, 4, 2, 1024, 128, 1),    # several units of an expert
    (17, 128, 1, 1, 8192, 0, 1),       # as many K steps as lanes
    (129, 1024, 3, 2, 128, 640, 2),    # two selections a lane, one token in the last workgroup, a longer shared expert
    (300, 512, 8, 3, 512, 0, 2),       # 126 selections
    (512, 512, 64, 2, 128, 128, 2),    # all that two lanes hold, and units on both sides
    (20, 512, 9, 26, 128, 0, 2),       # four tokens, selections of one in both of a lane's
]


@pytest.mark.parametrize("M,D,E,k,I,SI,lanes", SMALL_DOWN)
def test_small_layers_down_launch_gives_the_bits_of_down_and_combine(jg, M, D, E, k, I, SI, lanes):
    """Even routing, and one whose few experts have several units each; what a selection out of range leaves out."""
    for offset in (0, 20):
        test_small_layers_without_a_list_give_the_bits_of_the_sorted_rows(jg, M, D, E, min(k, E), I, SI, offset)
    if k > E:   # (a selection that is given may name an expert more than once)
        import torch
        params, rand = _layer(jg, D, E, I, 0, M)
        names = ("gate_proj", "up_proj", "down_proj")
        x, idx = rand(M, D), (torch.arange(M * k, device="cuda") * 7 % (E + 1)).int().reshape(M, k)   # (E: out of range)
        w = torch.rand(M, k, device="cuda")
        got = jg.expert_forward_single(x, idx, w, *(params[n] for n in names))
        parts = [jg.expert_forward_single(x, idx[:, s:s + 1].contiguous(), torch.ones(M, 1, device="cuda"), *(params[n] for n in names)) for s in range(k)]
        want = torch.zeros(M, D, device="cuda")
        for s in range(k):   # (one selection a token: its row in bf16)
            want = want + parts[s].float() * w[:, s:s + 1]
        assert torch.equal(got, want.bfloat16())


UNITS = [   # selections of each expert, D, E, k, I, SI
    ((8, 9, 16, 17, 7, 1), 256, 6, 1, 384, 0),        # whole and half units of h, an odd number of K steps
    ((24, 25, 1, 6, 8), 384, 9, 2, 128, 256),         # one K step; a shared expert; experts without rows
    ((33, 40, 8, 9, 2, 64, 124), 1024, 8, 2, 512, 0), # two selections a lane
]


@pytest.mark.parametrize("counts,D,E,k,I,SI", UNITS)
def test_small_layers_units_of_any_rows_give_the_grouped_bits(jg, counts, D, E, k, I, SI):
    """Units of 1 to 8, 9 to 15 and 16 rows, also where rows are zero or hold infinities and NaN, against the same tokens often enough
    for a sort."""
    import torch
    print("units of rows", counts, D, E, k, I, SI, flush=True)
    params, rand = _layer(jg, D, E, I, SI, D + I)
    names = ("gate_proj", "up_proj", "down_proj")
    same = lambda a, b: torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(7.0, float("inf"), -float("inf")), b.nan_to_num(7.0, float("inf"), -float("inf")))
    flat = np.repeat(np.arange(len(counts)), counts)
    M = len(flat) // k
    flat = H.rng_for(D).permutation(flat)[:M * k].reshape(M, k).astype(np.int32)
    idx, w = H.to_cuda(flat), torch.rand(M, k, device="cuda")
    for hard in (False, True):
        x = rand(M, D)
        if hard:
            x[0] = 0
            x[1, 5], x[2, 7], x[M - 1, D - 1] = float("inf"), float("nan"), -3e38
        if SI:   # (ready logits that select these: the chosen ones are the largest)
            lg = torch.full((M, E), -4.0, device="cuda").scatter_(1, (idx.long() + torch.arange(k, device="cuda") * 3) % E, 1.0)
            run = lambda n: jg.moe_experts(x.repeat(n, 1), lg.repeat(n, 1), top_k=k, experts={n_: params[n_] for n_ in names},
                                           shared={n_: params["shared_" + n_] for n_ in names})
        else:
            run = lambda n: jg.expert_forward_single(x.repeat(n, 1), idx.repeat(n, 1), w.repeat(n, 1), *(params[n_] for n_ in names))
        got, many = run(1), run(2048 // (M * k) + 1)
        assert same(got, many[:M]) and same(got, many[-M:])
        assert same(run(1), got)


@pytest.mark.parametrize("E,N,K,dtype", [(9, 2560, 2560, "bf16"), (9, 2560, 2688, "bf16"), (11, 2560, 2432, "f32"), (25, 512, 512, "f32")])   # two blocks wide; an odd number of blocks; sixteen waves; four, its experts eight
def test_large_weight_arrays_give_the_bits_of_their_experts(jg, E, N, K, dtype):
    import torch
    print("weight quantiser", E, N, K, dtype, flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(K)
    w = torch.randn(E, N, K, dtype=torch.bfloat16 if dtype == "bf16" else torch.float32, device="cuda", generator=gen)
    w[0, :128, :256] = 0                                     # all-zero blocks
    w[-1, -1, -1] = 1e30
    whole = jg.quantize_weight_block(w)
    for e in range(E):
        one = jg.quantize_weight_block(w[e])
        assert torch.equal(whole["w"][e].view(torch.uint8), one["w"].view(torch.uint8)) and torch.equal(whole["scale_inv"][e], one["scale_inv"]), e


@pytest.mark.parametrize("M,D,E,k,I,SI", [
    (3, 256, 8, 2, 384, 0),         # pairs of K steps in the first launch, an odd number of them in the second
    (2, 384, 8, 2, 256, 128),       # odd in the first, and in the second for the shared expert
    (5, 512, 8, 2, 512, 256),       # pairs in both
    (6, 2048, 128, 8, 768, 0),      # from memory: nine workgroups a CU in the first, 18 K steps a wave in the second
    (1, 7168, 18, 8, 2048, 2048),   # 1152 workgroups, 32 K steps
    (8, 1024, 8, 8, 1024, 0),       # from the caches, more workgroups in the first launch than the CUs hold of two K steps a stage
    (9, 512, 8, 2, 1024, 0),        # ... of short rows, more than four a CU
])
def test_single_tokens_in_stages_of_one_and_two_k_steps(jg, M, D, E, k, I, SI):
    test_experts_of_single_tokens_give_the_grouped_bits(jg, M, D, E, k, I, SI, False)


@pytest.mark.parametrize("E", [1, 17, 63, 64])
@pytest.mark.parametrize("rows", ["one", "few", "uneven", "alike", "large"])
def test_work_lists_of_one_wave_lead_to_the_same_rows(jg, E, rows):
    """Up to 64 experts are listed by one wave, 65 (the last ones without rows) by a workgroup: which item is whose differs, no
    row's bits do."""
    import torch
    print("one-wave list", E, rows, flush=True)
    D, I = 256, 128
    rng = H.rng_for(E)
    sizes = np.zeros(65, np.int64)
    sizes[:E] = {"one": 0, "few": rng.integers(0, 9, E), "uneven": rng.zipf(1.5, E).clip(0, 900) - 1, "alike": 40, "large": 13}[rows]
    if not sizes.any():
        sizes[E - 1] = 1
    if rows == "large":                 # beyond the last size class, 1023 x 32 rows
        sizes[E // 2] = 33000
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(E)
    rand = lambda *shape: torch.randn(*shape, dtype=torch.bfloat16, device="cuda", generator=gen)
    w = [jg.quantize_weight_block(rand(65, n, k).mul_(0.05)) for n, k in ((I, D), (I, D), (D, I))]
    xq, sx = jg.quant_act(rand(int(off[-1]), D))

    def rows_of(n):
        gate, up, down = ({"w": d["w"][:n].contiguous(), "scale_inv": d["scale_inv"][:n].contiguous()} for d in w)
        o = H.to_cuda(off[:n + 1].copy())
        hq, sh = jg.gemm_gateup_swiglu(xq, sx, gate, up, o)
        return hq.view(torch.uint8), sh, jg.gemm_down(hq, sh, down, o)

    for got, want in zip(rows_of(E), rows_of(65)):
        assert torch.equal(got, want)
