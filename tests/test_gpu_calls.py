"""The layer calls' native way (csrc/moe_call.cpp) against the general one: the same bits where it takes a call, and nothing
done where it does not."""
import gc

import numpy as np
import pytest

from tests.test_gpu_parity import jg  # noqa: F401

KEYS = ("gate_proj", "up_proj", "down_proj")


@pytest.fixture
def ways(jg, monkeypatch):
    """ways(call) -> (result of the native way, result of the general way), or the errors that they raise; and whether each
    call of the first went the native way."""
    from jax_gpt_amd import moe
    native = moe._native()

    class Watched:
        def __init__(self, take):
            self.take, self.taken = take, []

        def __getattr__(self, name):
            def call(*args):
                r = getattr(native, name)(*args) if self.take else None
                self.taken.append(r is not None)
                return r
            return call

    def both(call):
        out = []
        for take in (True, False):
            w = Watched(take)
            monkeypatch.setattr(moe, "_calls", w)
            try:
                out.append(call())
            except Exception as e:   # compared below
                out.append(e)
            if take:
                taken = w.taken
        return out[0], out[1], taken
    yield both
    gc.collect()   # (what the caught errors' frames still hold)


def _weights(jg, E, D, I, gen, names=KEYS):
    import torch
    q = lambda *s: jg.quantize_weight_block(torch.randn(s, dtype=torch.bfloat16, device="cuda", generator=gen).mul_(0.02))
    return dict(zip(names, (q(E, I, D), q(E, I, D), q(E, D, I))))


def _layer_params(jg, gen, D=256, E=8, I=128, SI=256):
    import torch
    p = _weights(jg, E, D, I, gen)
    p.update(_weights(jg, 1, D, SI, gen, tuple("shared_" + n for n in KEYS)))
    p["gate_weight"] = torch.randn(E, D, dtype=torch.bfloat16, device="cuda", generator=gen).t()
    p["shared_expert_gate_weight"] = torch.randn(1, D, dtype=torch.bfloat16, device="cuda", generator=gen).t()
    return p


def _same(a, b):
    import torch
    assert type(a) is type(b), (a, b)
    if isinstance(a, Exception):
        assert str(a) == str(b)
    elif isinstance(a, tuple):
        for x, y in zip(a, b):
            _same(x, y)
    else:
        assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [0, 1, 5, 40])
def test_calls_in_their_usual_form(jg, ways, M):
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M)
    D, E, I, k = 256, 8, 128, 2
    ex, p = _weights(jg, E, D, I, gen), _layer_params(jg, gen)
    shared = {n: p["shared_" + n] for n in KEYS}
    r = lambda *s: torch.randn(s, device="cuda", generator=gen)
    x, lg, norm = r(M, D).bfloat16(), r(M, E), r(D)
    x3 = x.reshape(1, M, D)
    calls = [lambda: jg.moe_experts(x, lg, top_k=k, experts=ex),
             lambda: jg.moe_experts(x, lg, top_k=k, experts=ex, routing="sigmoid_grouped", bias=norm[:E].clone(), n_group=4,
                                    topk_group=2, routed_scale=2.5, shared=shared, renorm=False),
             lambda: jg.moe_experts(x, None, top_k=k, experts=ex, shared=shared, gate_weight=p["gate_weight"],
                                    shared_expert_gate_weight=p["shared_expert_gate_weight"], norm_weight=norm, add_residual=True),
             lambda: jg.moe_layer(x3, p, k), lambda: jg.moe_layer(x3.float(), p, k),
             lambda: jg.moe_layer(x3, {n: v for n, v in p.items() if not n.startswith("shared")}, k),
             lambda: jg.moe_sublayer(x3, norm, p, k), lambda: jg.moe_sublayer(x3.float(), norm, p, k, 1e-3),
             lambda: jg.moe_routing(x, p["gate_weight"], k),
             lambda: jg.expert_forward_single(x, *jg.route_softmax_topk(lg, k), *(ex[n] for n in KEYS))]
    for i, call in enumerate(calls):
        a, b, taken = ways(call)
        assert taken == [True], i
        assert not isinstance(a, Exception), (i, a)
        _same(a, b)


@pytest.mark.gpu
def test_calls_in_other_forms_go_the_general_way(jg, ways):
    """Converted or refused there, as without the native way."""
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(7)
    M, D, E, I, k = 5, 256, 8, 128, 2
    ex, p = _weights(jg, E, D, I, gen), _layer_params(jg, gen)
    r = lambda *s: torch.randn(s, device="cuda", generator=gen)
    x, lg, norm = r(M, D).bfloat16(), r(M, E), r(D)
    x3 = x.reshape(1, M, D)
    plain = {n: r(E, I, D).transpose(1, 2) if n == "down_proj" else r(E, D, I) for n in KEYS}
    as_bytes = {n: dict(w=d["w"].view(torch.uint8), scale_inv=d["scale_inv"]) for n, d in ex.items()}
    thin = {n: dict(w=d["w"], scale_inv=d["scale_inv"][:, :, :1]) for n, d in ex.items()}
    odd = torch.empty(M * D + 1, device="cuda")[1:].view(1, M, D)
    odd.copy_(x3)
    calls = [lambda: jg.moe_experts(r(D, M).bfloat16().t()[:, :D], lg, top_k=k, experts=plain),
             lambda: jg.moe_experts(x, lg, top_k=k, experts=as_bytes),
             lambda: jg.moe_experts(x, lg.t().contiguous().t(), top_k=k, experts=ex),
             lambda: jg.moe_layer(odd, p, k), lambda: jg.moe_sublayer(x3, norm.bfloat16(), p, k),
             lambda: jg.moe_routing(x.t().contiguous().t(), p["gate_weight"].float(), k),
             # refused
             lambda: jg.moe_experts(x.float(), lg, top_k=k, experts=ex), lambda: jg.moe_experts(x3, lg, top_k=k, experts=ex),
             lambda: jg.moe_experts(x, lg[:3], top_k=k, experts=ex), lambda: jg.moe_experts(x, lg.cpu(), top_k=k, experts=ex),
             lambda: jg.moe_experts(x, lg, top_k=k, experts=thin), lambda: jg.moe_experts(x, lg, top_k=k, experts=dict(ex, up_proj=p["shared_up_proj"])),
             lambda: jg.moe_experts(x, lg, top_k=k, experts=ex, routing="none"), lambda: jg.moe_experts(x, None, top_k=k, experts=ex),
             lambda: jg.moe_experts(x, lg, top_k=k, experts=ex, gate_weight=p["gate_weight"]),
             lambda: jg.moe_experts(x, lg, top_k=k, experts=ex, shared_expert_gate_weight=p["shared_expert_gate_weight"]),
             lambda: jg.moe_layer(x, p, k), lambda: jg.moe_layer(x3.half(), p, k), lambda: jg.moe_layer(x3, dict(p, gate_weight=p["gate_weight"][:, :3]), k),
             lambda: jg.moe_sublayer(x3, norm[:9], p, k), lambda: jg.moe_routing(x, p["gate_weight"].t(), k),
             # refused by the library
             lambda: jg.moe_experts(x, lg, top_k=E + 1, experts=ex), lambda: jg.moe_layer(x3, p, -1)]
    for i, call in enumerate(calls):
        gen.manual_seed(i)
        state = gen.get_state()
        a, b, taken = ways(lambda: (gen.set_state(state), call())[1])
        if i < 21:
            assert not any(taken[:1]), i   # (the view at an odd offset is copied, and the copy is in the usual form)
        _same(a, b)
        if i >= 6:
            assert isinstance(a, Exception), (i, a)
    doubled = torch.vmap(lambda t: jg.moe_experts(t, lg, top_k=k, experts=ex))
    a, b, taken = ways(lambda: doubled(torch.stack([x, x])))
    assert not any(taken) and isinstance(a, Exception) and type(a) is type(b)


@pytest.mark.gpu
def test_calls_with_other_scalars_go_the_general_way(jg, ways):
    """Calls that differ from a taken one in the type of one number alone: converted, or refused, as without the native way."""
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(11)
    M, D, E, I, k = 5, 256, 8, 128, 2
    ex, p = _weights(jg, E, D, I, gen), _layer_params(jg, gen)
    r = lambda *s: torch.randn(s, device="cuda", generator=gen)
    x, lg, norm = r(M, D).bfloat16(), r(M, E), r(D)
    base = dict(top_k=k, experts=ex, routing="sigmoid_grouped", n_group=4, topk_group=2, renorm=True, routed_scale=2.5, norm_weight=norm, norm_eps=1e-6,
                add_residual=True)
    whole = (lambda **kw: jg.moe_experts(x, lg, **dict(base, **kw)))
    a, b, taken = ways(whole)
    assert taken == [True] and not isinstance(a, Exception)
    _same(a, b)
    for kw in (dict(top_k=np.int64(k)), dict(top_k=2.0), dict(top_k="2"), dict(top_k=None), dict(top_k=1 << 40), dict(n_group=np.int32(4)), dict(topk_group=2.0),
               dict(renorm=np.bool_(True)), dict(renorm=1.0), dict(routed_scale=2), dict(routed_scale=np.float32(2.5)), dict(norm_eps=0), dict(norm_eps=np.float64(1e-6)),
               dict(add_residual=np.bool_(True))):
        a, b, taken = ways(lambda: whole(**kw))
        assert taken == [False], kw
        _same(a, b)
    for call in (lambda: jg.moe_routing(x, p["gate_weight"], np.int64(k)), lambda: jg.moe_layer(x[None], p, np.int32(k)),
                 lambda: jg.moe_sublayer(x[None], norm, p, k, 0)):
        a, b, taken = ways(call)
        assert not any(taken)
        _same(a, b)


def test_native_way_takes_nothing_from_the_cpu():
    """Without a GPU: every entry point of the module declines, and reads no address it was bound to."""
    import ctypes
    import torch
    from jax_gpt_amd import moe, moe_call
    if moe._calls is not None:
        pytest.skip("bound to the library: runs where no GPU is")
    hit = ctypes.CFUNCTYPE(ctypes.c_int)(lambda: pytest.fail("a declined call reached the library"))
    at = ctypes.cast(hit, ctypes.c_void_p).value
    moe_call.bind(*[at] * 6, pytest.fail, pytest.fail, pytest.fail, pytest.fail)
    x = torch.zeros(4, 256, dtype=torch.bfloat16)
    d = {n: dict(w=torch.zeros(8, *s, dtype=torch.float8_e4m3fn), scale_inv=torch.zeros(8, s[0] // 128, s[1] // 128))
         for n, s in zip(KEYS, ((128, 256), (128, 256), (256, 128)))}
    tail = (0, None, 1, 1, 1, 1.0, None, None, None, None, 1e-6, 0, 0, None, 2)
    for v in (x, x.float().numpy(), None, torch.nn.Parameter(x)):
        assert moe_call.experts(v, torch.zeros(4, 8), 2, d, *tail) is None
        assert moe_call.layer(v, dict(d, gate_weight=x.t()), 2, None, 1e-6, 0) is None
        assert moe_call.routing(v, x.t(), 2) is None
    for bad in (np.int64(2), 2.0, "2", None, 1 << 40):
        assert moe_call.experts(x, torch.zeros(4, 8), bad, d, *tail) is None and moe_call.routing(x, x.t(), bad) is None
    assert moe_call.experts() is None and moe_call.layer(x) is None and moe_call.routing(x, x) is None
    with pytest.raises(ValueError):
        moe_call.bind(*[0] * 6, None, None, None, None)
