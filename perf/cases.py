"""The work that users of this package have it do, as measurable cases.

Every case is one pass through the public entry points of `jax_gpt_amd`:

* `experts`    router logits in, combined hidden states out (`moe_experts`): benchmark configurations 1 to 4
* `functions`  the reference's functions called one by one (`moe_routing`, then `expert_forward_single`)
* `layer`      hidden states in, with the router and the gated shared expert (`moe_layer`), bf16 or f32 activations
* `sublayer`   the same between the block's RMSNorm and its residual add (`moe_sublayer`)
* `shard`      one GPU's expert-parallel share of rows that another GPU dispatched (benchmark configuration 5)
* `quantize`   bf16 or f32 checkpoint weights to block-scaled fp8 (`quantize_weight_block`), what loading a layer costs

The layers are the ones of the benchmark configurations and of the presets that the tests use; weights, activations
and logits have the benchmark's distributions.
"""
import functools
import math

import numpy as np
import torch

import jax_gpt_amd as jg

# hidden size, routed experts, experts per token, expert intermediate size, shared intermediate size, routing
LAYERS = {
    "tiny": dict(D=512, E=8, k=2, I=1024, SI=0, routing="softmax"),                        # benchmark configuration 1
    "mini": dict(D=1024, E=32, k=2, I=512, SI=512, routing="softmax"),                     # the mini preset
    "qwen3": dict(D=2048, E=128, k=8, I=768, SI=0, routing="softmax"),                     # configuration 2
    "full": dict(D=4096, E=512, k=10, I=1024, SI=1024, routing="softmax"),                 # the full preset
    "deepseek": dict(D=7168, E=256, k=8, I=2048, SI=2048, routing="sigmoid_grouped"),      # configurations 3 and 4
}
GROUPS = dict(n_group=8, topk_group=4)     # the group-limited router of the DeepSeek-V3 layer
BIAS_STD = 0.1
SHARD = dict(D=7168, E=32, k=8, I=2048)    # configuration 5: 32 local experts of the DeepSeek-V3 layer


def listed():
    return [
        # a toy layer, as in a first test or a debugging run: launches and host work
        dict(name="tiny layer, 256 tokens", entry="experts", layer="tiny", tokens=256),
        # one stream generating text with a small model: the smallest call there is
        dict(name="mini sublayer, 1 token", entry="sublayer", layer="mini", tokens=1, x="bf16"),
        # one stream generating text with the largest layer: eight experts' weights are read
        dict(name="deepseek decode, 1 token", entry="experts", layer="deepseek", tokens=1),
        # a serving batch in decode: half of the experts' weights are read for one or two rows each
        dict(name="deepseek decode, 64 tokens", entry="experts", layer="deepseek", tokens=64),
        # a chunk of a prompt beside other requests: every expert has a few rows
        dict(name="deepseek chunk, 777 tokens", entry="experts", layer="deepseek", tokens=777),
        # a full prompt batch, the headline of the benchmark
        dict(name="deepseek prefill, 8192 tokens", entry="experts", layer="deepseek", tokens=8192),
        # a decode batch through the reference's own functions
        dict(name="qwen3 functions, 33 tokens", entry="functions", layer="qwen3", tokens=33),
        # a prompt batch of the smaller production layer
        dict(name="qwen3 prefill, 4096 tokens", entry="experts", layer="qwen3", tokens=4096),
        # a decode batch through the whole half block: norm, router, experts, gated shared expert, residual
        dict(name="full sublayer, 32 tokens", entry="sublayer", layer="full", tokens=32, x="bf16"),
        # a prompt of odd length from a caller that keeps its activations in f32
        dict(name="full layer f32, 2047 tokens", entry="layer", layer="full", tokens=2047, x="f32"),
        # an expert-parallel rank: rows arrive grouped by expert, very unevenly, some experts get none
        dict(name="shard, 16384 rows", entry="shard", tokens=2048),
        # loading: sixteen experts' worth of one projection at a time
        dict(name="quantize bf16, 16 experts", entry="quantize", experts=16, out=2048, inner=7168, x="bf16"),
    ]


def _log_between(rng, lo, hi):
    """A whole number, its logarithm evenly spread."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo - 0.49), math.log(hi + 0.49)))))))


def draw(rng):
    entry = rng.choice(["experts", "experts", "experts", "functions", "layer", "sublayer", "shard", "quantize"])
    if entry == "experts":
        layer = rng.choice(["tiny", "qwen3", "deepseek", "deepseek"])
        return dict(entry=entry, layer=layer, tokens=_log_between(rng, 1, 4096 if layer == "qwen3" else 8192))
    if entry == "functions":
        return dict(entry=entry, layer=rng.choice(["tiny", "qwen3"]), tokens=_log_between(rng, 1, 4096))
    if entry in ("layer", "sublayer"):
        return dict(entry=entry, layer=rng.choice(["mini", "full"]), tokens=_log_between(rng, 1, 4096), x=rng.choice(["bf16", "f32"]))
    if entry == "shard":
        return dict(entry=entry, tokens=_log_between(rng, 8, 2048))
    return dict(entry=entry, experts=_log_between(rng, 1, 16), out=128 * rng.randint(4, 56), inner=128 * rng.randint(4, 56),
                x=rng.choice(["bf16", "f32"]))


# ---- inputs ----

def _randn(shape, gen, std=1.0, dtype=torch.bfloat16):
    t = torch.randn(shape, dtype=dtype, device="cuda", generator=gen)
    return t if std == 1.0 else t.mul_(std)


def _fp8(E, N, K, gen, chunk=32):
    """(E, N, K) N(0, 0.02) weights, block-quantised a few experts at a time."""
    wq = torch.empty((E, N, K), dtype=torch.float8_e4m3fn, device="cuda")
    sw = torch.empty((E, N // 128, K // 128), dtype=torch.float32, device="cuda")
    for e in range(0, E, chunk):
        d = jg.quantize_weight_block(_randn((min(chunk, E - e), N, K), gen, 0.02))
        wq[e:e + chunk], sw[e:e + chunk] = d["w"], d["scale_inv"]
    return {"w": wq, "scale_inv": sw}


def _swiglu(E, D, I, gen, names=("gate_proj", "up_proj", "down_proj")):
    return dict(zip(names, (_fp8(E, I, D, gen), _fp8(E, I, D, gen), _fp8(E, D, I, gen))))


def _group_sizes(R, seed):
    """Zipf(1.2) over the local experts, three of them without rows."""
    E = SHARD["E"]
    rng = np.random.default_rng(seed)
    p = 1.0 / np.arange(1, E + 1) ** 1.2
    p[[5, 17, 30]] = 0.0
    return rng, np.bincount(rng.choice(E, size=R, p=p / p.sum()), minlength=E).astype(np.int32)


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    entry = case["entry"]
    if entry == "quantize":
        dtype = torch.float32 if case["x"] == "f32" else torch.bfloat16
        return dict(entry=entry, w=_randn((case["experts"], case["out"], case["inner"]), gen, 0.02, dtype))
    M = case["tokens"]
    if entry == "shard":
        D, E, k, I = (SHARD[n] for n in ("D", "E", "k", "I"))
        R = M * k
        rng, sizes = _group_sizes(R, seed)
        offsets = torch.from_numpy(np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)).cuda()
        xq, sx = jg.quant_act(_randn((R, D), gen))          # rows arrive quantised, as the dispatch sends them
        return dict(entry=entry, experts=_swiglu(E, D, I, gen), xq=xq, sx=sx, offsets=offsets,
                    weights=torch.from_numpy(rng.dirichlet(np.ones(k), size=M).astype(np.float32)).cuda(),
                    inv_perm=torch.from_numpy(rng.permutation(R).astype(np.int32)).cuda())
    L = LAYERS[case["layer"]]
    D, E, k, I, SI = (L[n] for n in ("D", "E", "k", "I", "SI"))
    if entry in ("layer", "sublayer"):
        params = _swiglu(E, D, I, gen)
        params.update(_swiglu(1, D, SI, gen, ("shared_gate_proj", "shared_up_proj", "shared_down_proj")))
        # router weights as a checkpoint holds them, (out, in), seen through a transposed view
        params["gate_weight"] = _randn((E, D), gen, 0.02).t()
        params["shared_expert_gate_weight"] = _randn((1, D), gen, 0.02).t()
        x = _randn((1, M, D), gen, dtype=torch.float32 if case["x"] == "f32" else torch.bfloat16)
        return dict(entry=entry, params=params, k=k, x=x, norm=_randn((D,), gen, 0.1, torch.float32))
    state = dict(entry=entry, experts=_swiglu(E, D, I, gen), k=k, x=_randn((M, D), gen))
    if entry == "functions":
        state["gate_weight"] = _randn((E, D), gen, 0.02).t()
        return state
    state["logits"] = _randn((M, E), gen, dtype=torch.float32)
    state["kw"] = dict(routing=L["routing"])
    if L["routing"] == "sigmoid_grouped":
        state["kw"].update(GROUPS, bias=_randn((E,), gen, BIAS_STD, torch.float32))
    if SI:
        state["kw"]["shared"] = _swiglu(1, D, SI, gen)
    return state


# ---- one pass ----

def run(state):
    s, entry = state, state["entry"]
    if entry == "experts":
        return jg.moe_experts(s["x"], s["logits"], top_k=s["k"], experts=s["experts"], **s["kw"])
    if entry == "functions":
        idx, w = jg.moe_routing(s["x"], s["gate_weight"], s["k"])
        e = s["experts"]
        return jg.expert_forward_single(s["x"], idx, w, e["gate_proj"], e["up_proj"], e["down_proj"])
    if entry == "layer":
        return jg.moe_layer(s["x"], s["params"], s["k"])
    if entry == "sublayer":
        return jg.moe_sublayer(s["x"], s["norm"], s["params"], s["k"])
    if entry == "shard":
        e = s["experts"]
        scales = jg.gather_scales(s["sx"])
        hq, sh = jg.gemm_gateup_swiglu(s["xq"], scales, e["gate_proj"], e["up_proj"], s["offsets"], block_major=True)
        y = jg.gemm_down(hq, sh, e["down_proj"], s["offsets"], block_major=True)
        return jg.combine(y, s["weights"], s["inv_perm"])
    d = jg.quantize_weight_block(s["w"])
    return d["w"].view(torch.uint8), d["scale_inv"]


# ---- what a pass cannot do without ----

@functools.lru_cache(maxsize=None)
def _touched(layer, M):
    """Experts that get at least one row of M tokens: counted on one draw of the benchmark's router inputs."""
    L = LAYERS[layer]
    E, k = L["E"], L["k"]
    if L["routing"] == "softmax":        # every expert is as likely as the next
        return E * (1.0 - (1.0 - k / E) ** M)
    rng = np.random.default_rng(0)
    n, keep = GROUPS["n_group"], GROUPS["topk_group"]
    bias = rng.standard_normal(E) * BIAS_STD
    seen = np.zeros(E, bool)
    for _ in range(0, M, 1024):
        m = min(M, 1024)
        score = 1.0 / (1.0 + np.exp(-rng.standard_normal((m, E)))) + bias
        groups = score.reshape(m, n, E // n)
        best = np.argsort(-np.sort(groups, axis=2)[:, :, -2:].sum(2), axis=1)[:, :keep]
        kept = np.full_like(groups, -np.inf)
        rows = np.arange(m)[:, None]
        kept[rows, best] = groups[rows, best]
        seen[np.argpartition(-kept.reshape(m, E), k, axis=1)[:, :k].ravel()] = True
    return float(seen.sum())


def _expert_bytes(D, I):
    return 3 * D * I + 3 * (D // 128) * (I // 128) * 4


def work(case):
    """Each input read once (of the experts: those that have rows), each output written once; products counted as
    two operations per multiplication."""
    entry = case["entry"]
    if entry == "quantize":
        n = case["experts"] * case["out"] * case["inner"]
        return {"bytes": n * ((4 if case["x"] == "f32" else 2) + 1 + 4 / 128 ** 2), "flops": 0}
    M = case["tokens"]
    if entry == "shard":
        D, I, k = SHARD["D"], SHARD["I"], SHARD["k"]
        R = M * k
        touched = int((_group_sizes(R, 0)[1] > 0).sum())
        return {"bytes": touched * _expert_bytes(D, I) + R * (D + D // 128 * 4 + 8) + M * D * 2, "flops": 6.0 * R * D * I}
    L = LAYERS[case["layer"]]
    D, E, k, I, SI = (L[n] for n in ("D", "E", "k", "I", "SI"))
    size = 4 if case.get("x") == "f32" else 2
    b = _touched(case["layer"], M) * _expert_bytes(D, I) + 2 * M * D * size
    f = 6.0 * M * k * D * I
    if SI:
        b += _expert_bytes(D, SI)
        f += 6.0 * M * D * SI
    if entry == "experts":
        b += M * E * 4
    else:
        b += E * D * 2
        f += 2.0 * M * D * E
    return {"bytes": b, "flops": f}


def tolerance(case):
    """fp8 products and bf16 results (e4m3 rounding boundaries are crossed on a few in a thousand of the intermediate
    values).  Where the router's bf16 logits are computed inside, equal or neighbouring logits may also swap the last
    expert of a token or two."""
    if case["entry"] == "quantize":
        return "exact"
    if case["entry"] in ("functions", "layer", "sublayer"):
        return {"rel": 2e-2, "max": 0.9}
    return {"rel": 1e-2, "max": 0.2}
