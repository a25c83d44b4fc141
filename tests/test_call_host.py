"""The native host work of the layer calls (csrc/moe_call.cpp) without a GPU: the module built to take CPU tensors, over a library
that records what it is called with."""
import ctypes as C
import importlib.machinery
import importlib.util
import os
import shutil
import subprocess
import sys
import types
import weakref

import numpy as np
import pytest
import torch

from jax_gpt_amd import _lib
from tests.test_gpu_calls import KEYS

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _build_module():
    spec = importlib.util.spec_from_file_location("_call_build", os.path.join(ROOT, "jax-gpt_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    return build


@pytest.fixture(scope="module")
def module(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs a C++ compiler")
    build = _build_module()
    out = tmp_path_factory.mktemp("call")
    source, so = str(out / "host.cpp"), str(out / "moe_call.so")
    headers = [line for line in open(os.path.join(build.CSRC, "moe_call.cpp")) if line.startswith("#include <")]
    with open(source, "w") as f:   # (torch's headers first: the substitution reaches the module's own text alone)
        f.write("".join(headers) + f'#define is_cuda is_cpu\n#include "{os.path.join(build.CSRC, "moe_call.cpp")}"\n')
    command = build._call_command()
    command[command.index(os.path.join(build.CSRC, "moe_call.cpp"))] = source
    command[command.index("-o") + 1] = so
    subprocess.run(command, check=True)
    loader = importlib.machinery.ExtensionFileLoader("moe_call", so)
    module = importlib.util.module_from_spec(importlib.util.spec_from_file_location("moe_call", so, loader=loader))
    loader.exec_module(module)
    return module


class Library:
    """The functions that moe_call is bound to.  Every forward call's arguments are appended to `calls`."""

    def __init__(self, module, router_weight=None):
        self.calls, self.codes = [], []
        size = C.CFUNCTYPE(C.c_size_t, *[C.c_int] * 6)(lambda *a: 64)
        forward = C.CFUNCTYPE(C.c_int, C.POINTER(_lib.MoeForwardArgs), C.c_void_p, C.c_size_t, C.c_void_p)(self._forward)
        selected = C.CFUNCTYPE(C.c_int, C.POINTER(_lib.MoeForwardArgs), *[C.c_void_p] * 3, C.c_size_t, C.c_void_p)(self._forward)
        router_size = C.CFUNCTYPE(C.c_size_t, *[C.c_int] * 3)(lambda *a: 64)
        routing = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_int, C.c_int, C.c_void_p, *[C.c_int] * 3, *[C.c_void_p] * 3, C.c_size_t, C.c_void_p)(
            lambda *a: self.calls.append(a) or 0)
        self.bound = size, forward, forward, selected, router_size, routing
        module.bind(*(C.cast(f, C.c_void_p).value for f in self.bound), self.codes.append, router_weight or self._router_weight,
                    lambda: 0, lambda device: 0)

    def _forward(self, args, *rest):
        got = _lib.MoeForwardArgs()
        C.pointer(got)[0] = args[0]
        self.calls.append(got)
        return 0

    @staticmethod
    def _router_weight(w, name):
        return w.t().contiguous()


def _layer_params(D=256, E=8, I=128, SI=256):
    def fp8(e, n, k):
        return dict(w=torch.zeros(e, n, k, dtype=torch.float8_e4m3fn), scale_inv=torch.ones(e, n // 128, k // 128))
    p = dict(zip(KEYS, (fp8(E, I, D), fp8(E, I, D), fp8(E, D, I))))
    p.update(zip(("shared_" + n for n in KEYS), (fp8(1, SI, D), fp8(1, SI, D), fp8(1, D, SI))))
    p["gate_weight"] = torch.zeros(E, D, dtype=torch.bfloat16).t()
    p["shared_expert_gate_weight"] = torch.zeros(1, D, dtype=torch.bfloat16).t()
    return p


def test_router_weights_outlive_their_dict_entries(module):
    """Fetching the router weight runs Python code; the shared expert's gate, which the dict alone may hold and which comes next, has
    to outlive what that code, or another thread meanwhile, does to the dict."""
    p = _layer_params()
    old = {n: weakref.ref(p[n]) for n in ("gate_weight", "shared_expert_gate_weight")}
    seen = []

    def fetch(w, name):
        if name == "gate_weight":
            for n in old:
                p[n] = torch.ones_like(old[n]())
            if old["shared_expert_gate_weight"]() is None:
                raise RuntimeError("freed while the call still needs it")   # (so that the call does not go on to read it)
        assert w is old[name]()
        seen.append(name)
        return w.t().contiguous()

    lib = Library(module, fetch)
    x = torch.zeros(1, 5, 256, dtype=torch.bfloat16)
    assert module.layer(x, p, 2, None, 1e-6, 0).shape == x.shape
    assert seen == list(old) and len(lib.calls) == 1 and lib.calls[0].w_shared_gate
    assert all(r() is None for r in old.values())   # (nor are they kept)


@pytest.mark.parametrize("there", [None, types.SimpleNamespace(__file__="old"),
                                   types.SimpleNamespace(__file__="struct", args_bytes=C.sizeof(_lib.MoeForwardArgs) - 8, torch_version=torch.__version__),
                                   types.SimpleNamespace(__file__="torch", args_bytes=C.sizeof(_lib.MoeForwardArgs), torch_version="1.13.0")],
                         ids=["missing", "without versions", "another struct", "another torch"])
def test_layer_calls_go_on_without_the_extension(lib, monkeypatch, there):
    """The general way needs the library alone: where the extension is not there, or of another build, it is said once and every
    call goes that way."""
    from jax_gpt_amd import moe
    monkeypatch.setitem(sys.modules, moe.__package__ + ".moe_call", there)
    package = sys.modules[moe.__package__]
    if there is None:
        monkeypatch.delattr(package, "moe_call", raising=False)
    else:
        monkeypatch.setattr(package, "moe_call", there, raising=False)
    monkeypatch.setattr(moe, "_calls", None)
    with pytest.warns(RuntimeWarning, match="in Python"):
        calls = moe._native()
    assert calls.layer(0, 0, 0, 0, 0, 0) is calls.routing(0, 0, 0) is calls.experts(*range(19)) is None
    assert moe._native() is calls


@pytest.mark.parametrize("trouble", ["no torch", "no compiler", "compile error"])
def test_the_library_is_linked_whatever_becomes_of_the_extension(monkeypatch, tmp_path, trouble):
    """The compilers' calls alone: only the extension's may fail, or be missing, and the library is linked before it."""
    build, ran = _build_module(), []

    class Process:
        returncode = 0

        def __init__(self, command, **kw):
            ran.append(command)
            if "-lc10" in command:
                if trouble == "no compiler":
                    raise FileNotFoundError(command[0])
                self.returncode = 1

        def communicate(self):
            return "", None

    monkeypatch.setattr(build, "HERE", str(tmp_path))
    monkeypatch.setattr(build, "_hipcc", lambda: "hipcc")
    monkeypatch.setattr(build.subprocess, "Popen", Process)
    monkeypatch.setattr(build.subprocess, "run", lambda command, check: ran.append(command))
    if trouble == "no torch":
        monkeypatch.setitem(sys.modules, "torch", None)
        assert build.build(verbose=False) == build.LIB_PATH
    else:
        with pytest.raises((RuntimeError, FileNotFoundError)):
            build.build(verbose=False)
    links = [i for i, c in enumerate(ran) if c[-1] == build.LIB_PATH]
    assert len(links) == 1 and all(i > links[0] for i, c in enumerate(ran) if "-lc10" in c)


class OnGpu(torch.Tensor):
    is_cuda = property(lambda self: True)


def on_gpu(t):
    return {k: on_gpu(v) for k, v in t.items()} if isinstance(t, dict) else t.as_subclass(OnGpu)


@pytest.fixture
def general(monkeypatch):
    """moe.py whose extension declines every call (the names of its functions that were called) and whose library does nothing."""
    from jax_gpt_amd import moe
    offered = []

    class Declines:
        def __getattr__(self, name):
            return lambda *args: offered.append(name)

    class NoLibrary:
        moe_forward_workspace_bytes = staticmethod(lambda *a: 64)
        moe_forward = moe_forward_f32 = staticmethod(lambda *a: 0)

    monkeypatch.setattr(moe, "_calls", Declines())
    monkeypatch.setattr(moe, "lib", NoLibrary)
    monkeypatch.setattr(moe, "_stream", lambda: 0)
    return moe, offered


def test_layer_calls_in_other_forms_are_offered_once(general):
    """A call that the extension does not take is declined once, not again on the general way."""
    moe, offered = general
    p = on_gpu(_layer_params())
    x, norm = on_gpu(torch.zeros(1, 5, 256, dtype=torch.bfloat16)), on_gpu(torch.zeros(256))
    for call in (lambda: moe.moe_layer(x, p, 2), lambda: moe.moe_sublayer(x, norm, p, 2), lambda: moe.moe_layer(on_gpu(x.float()), p, 2),
                 lambda: moe.moe_experts(x[0], on_gpu(torch.zeros(5, 8)), top_k=2, experts=p)):
        offered.clear()
        assert call().shape[-1] == 256 and len(offered) == 1, offered


def test_a_selection_bias_holds_a_value_an_expert(module, general):
    """A shorter one is refused, not read beyond its end; softmax routing reads none, and a longer one's end is not read."""
    moe, _ = general
    lib, p, E = Library(module), _layer_params(), 8
    x, logits = torch.zeros(5, 256, dtype=torch.bfloat16), torch.zeros(5, E)

    def native(bias, routing):
        return module.experts(x, logits, 2, p, routing, bias, 1, 1, 1, 1.0, None, None, None, None, 1e-6, 0, 0, None, 2)

    def python(bias, routing):
        return moe.moe_experts(on_gpu(x), on_gpu(logits), top_k=2, experts=on_gpu(p), routing=routing, bias=on_gpu(bias))
    for n in (0, E - 1):
        assert native(torch.zeros(n), 1) is None and not lib.calls
        with pytest.raises(ValueError, match="bias"):
            python(torch.zeros(n), "sigmoid_grouped")
        assert python(torch.zeros(n), "softmax").shape == x.shape
    for n in (E, E + 1):
        assert native(torch.zeros(n), 1).shape == python(torch.zeros(n), "sigmoid_grouped").shape == x.shape
    assert len(lib.calls) == 2


@pytest.mark.parametrize("at,value", [(2, np.int64(2)), (2, 2.0), (2, "2"), (2, None), (2, 1 << 40), (2, -(1 << 40)), (4, 0.0), (6, np.int32(4)), (7, None),
                                      (8, np.bool_(True)), (9, 2), (9, np.float32(2.5)), (14, 0), (14, np.float64(1e-6)), (15, np.bool_(True)), (16, None),
                                      (18, 2.0), (18, 4)])
def test_other_scalars_are_declined(module, at, value):
    """A call that is taken, and the same with one number of another type, or beyond an int."""
    lib, x = Library(module), torch.zeros(5, 256, dtype=torch.bfloat16)
    call = [x, torch.zeros(5, 8), 2, _layer_params(), 1, None, 4, 2, True, 2.5, None, None, None, torch.zeros(256), 1e-6, True, False, None, 2]
    assert module.experts(*call).shape == x.shape and len(lib.calls) == 1
    a = lib.calls.pop()
    assert (a.M, a.D, a.E, a.k, a.I, a.SI, a.routing, a.n_group, a.topk_group, a.renorm, a.routed_scale, a.add_residual) == (5, 256, 8, 2, 128, 0, 1, 4, 2, 1, 2.5, 1)
    assert a.norm_eps == np.float32(1e-6) and a.x == x.data_ptr()
    call[at] = value
    assert module.experts(*call) is None and not lib.calls
    if at == 2:
        p = _layer_params()
        assert module.routing(x, p["gate_weight"], 2) and len(lib.calls) == 1
        assert module.routing(x, p["gate_weight"], value) is None and len(lib.calls) == 1
        assert module.layer(x[None], p, 2, None, 1e-6, 0) is not None and len(lib.calls) == 2
        assert module.layer(x[None], p, value, None, 1e-6, 0) is None and len(lib.calls) == 2
