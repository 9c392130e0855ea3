"""The MLP under torch's transforms (CPU, the extension stubbed): F.silu(gate) *
up (runtime/llama.py:253-256) runs as one raw-pointer launch only where nothing
but eager execution sees it.  Gradients, forward-mode tangents, vmap and traces
of an MLP over plain tensors, and of one over quantized weights whose chunk takes
the dequant + F.linear route, are torch's own; a plain tensor's MLP never
reaches the launch."""

import pytest
import torch
import torch.nn.functional as F
from torch.autograd import forward_ad
from torch.fx.experimental.proxy_tensor import make_fx

from gdsllm_amd.runtime import llama, qwen_moe

H, FFN, T = 32, 96, 5


class Ext:
    """The dequant route on the CPU, and a silu_mul that loses what a raw-pointer
    launch loses: everything but the values."""

    def __init__(self):
        self.launches = 0

    def dequant_gguf(self, w, shape, gguf_type, offset, scratch):
        return w

    def silu_mul(self, gate, up):
        self.launches += 1
        return torch.from_numpy((F.silu(gate) * up).numpy())


@pytest.fixture
def ext(monkeypatch):
    e = Ext()
    monkeypatch.setattr(llama, "ext", lambda: e)
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)  # so that only the rules under test decide
    return e


def _weights(quantized):
    g = torch.Generator().manual_seed(1)
    out = {}
    for name, shape in (("gate", (FFN, H)), ("up", (FFN, H)), ("down", (H, FFN))):
        w = (torch.randn(shape, generator=g) * 0.2).half()
        out[f"mlp.{name}_proj.weight"] = \
            {"buffer": w, "shape": list(shape), "gguf_type": "q5_k", "offset": 0} if quantized else w
    return out


def _reference(x, weights):
    g, u, d = (w["buffer"] if isinstance(w, dict) else w for w in weights.values())
    return F.linear(F.silu(F.linear(x, g)) * F.linear(x, u), d)


class _Buf:
    device_id = 0


def _x(seed=2):
    return torch.randn(1, T, H, generator=torch.Generator().manual_seed(seed)).half()


@pytest.fixture(params=[False, True], ids=["plain", "quantized"])
def mlp(request, ext, monkeypatch):
    weights = _weights(request.param)
    monkeypatch.setattr(llama, "_gguf_pair", lambda g, u: False)  # stub buffers have no device
    return (lambda x: llama.mlp(x, weights)), (lambda x: _reference(x, weights)), ext, request.param


def test_eager(mlp):
    """The launch serves quantized weights only."""
    run, want, ext, quantized = mlp
    assert torch.equal(run(_x()), want(_x()))
    assert ext.launches == (1 if quantized else 0)


def test_forward_mode(mlp):
    run, want, _, _ = mlp
    with forward_ad.dual_level():
        tangents = [forward_ad.unpack_dual(f(forward_ad.make_dual(_x(), _x(3)))).tangent for f in (run, want)]
        assert tangents[0] is not None and torch.equal(*tangents)


def test_func_jvp(mlp):
    run, want, _, _ = mlp
    got, ref = (torch.func.jvp(f, (_x(),), (_x(3),)) for f in (run, want))
    assert torch.equal(got[0], ref[0]) and torch.equal(got[1], ref[1])


def test_gradient(mlp):
    run, want, _, _ = mlp
    grads = []
    for f in (run, want):
        x = _x().requires_grad_()
        f(x).float().sum().backward()
        grads.append(x.grad)
    assert torch.equal(*grads)


def test_vmap(mlp):
    run, want, _, _ = mlp
    x = torch.stack([_x(4), _x(5), _x(6)])
    assert torch.equal(torch.func.vmap(run)(x), torch.func.vmap(want)(x))


@pytest.mark.parametrize("trace", [lambda f, x: torch.jit.trace(f, x, check_trace=False), lambda f, x: make_fx(f)(x)],
                         ids=["jit", "fx"])
def test_traces(mlp, trace):
    """A trace computes with the inputs it is called on."""
    run, want, ext, _ = mlp
    traced = trace(run, _x())
    assert torch.equal(traced(_x(7)), want(_x(7)))
    assert ext.launches == 0


def test_shared_expert_gate_up_is_eager_only(monkeypatch):
    """The fused gate/up/SiLU launch of a shared expert is refused to a
    transformed x (the separate projections then run)."""
    calls = []

    class Fused:
        def fused_affine_gate_up_silu_gemm(self, x, entries):
            calls.append(x)
            return x

    monkeypatch.setattr(qwen_moe, "ext", lambda: Fused())
    meta = {"buffer": _Buf(), "shape": [FFN, H], "quant_type": "affine_q4", "weight_offset": 0, "scale_offset": 0,
            "bias_offset": 0, "group_size": 32}
    weights = {f"mlp.shared_expert.{p}_proj.weight": dict(meta) for p in ("gate", "up")}
    fused = lambda x: qwen_moe._shared_gate_up_silu(x, weights)  # noqa: E731
    assert fused(_x()) is not None and len(calls) == 1
    with forward_ad.dual_level():
        assert fused(forward_ad.make_dual(_x(), _x(3))) is None
    assert fused(_x().requires_grad_()) is None
    refused = []
    torch.func.vmap(lambda x: refused.append(fused(x)) or x)(torch.stack([_x(4), _x(5)]))
    assert refused == [None] and len(calls) == 1
