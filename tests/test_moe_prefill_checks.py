"""mie_moe_prefill's argument checks and the MoE layer's choice of path, on the CPU."""

import pytest
import torch

from moe_engine import _native, fused_moe
from moe_engine.model import MoEFeedForward

INVALID, UNSUPPORTED, WORKSPACE = 1, 2, 3
F32, BF16, F64 = 0, 1, 3
GOOD = dict(x=1 << 24, tokens=33, ln_w=None, ln_b=None, eps=1e-5, residual=None, router=2 << 24, w1=3 << 24, b1=4 << 24, w2=5 << 24, b2=6 << 24, experts=8, top_k=2,
            dim=64, hidden=128, out=7 << 24, ws=8 << 24, ws_bytes=1 << 40, dtype=F32, stream=None)


@pytest.mark.parametrize(
    "change,status",
    [
        (dict(tokens=0), INVALID), (dict(experts=65), INVALID), (dict(top_k=9), INVALID),
        (dict(experts=1, top_k=2), INVALID), (dict(dim=66), INVALID), (dict(hidden=0), INVALID),
        (dict(dim=68, dtype=BF16), INVALID), (dict(dtype=F64), UNSUPPORTED), (dict(x=0), INVALID),
        (dict(w2=(5 << 24) + 8), INVALID), (dict(out=(7 << 24) + 4), INVALID), (dict(ws_bytes=64), WORKSPACE),
        (dict(ln_b=9 << 24), INVALID),
    ],
)
def test_bad_arguments_fail_before_launch(change, status):
    assert _native.lib().mie_moe_prefill(*{**GOOD, **change}.values()) == status
    assert _native.lib().mie_last_error()


def test_workspace_covers_the_last_chunk():
    lib = _native.lib()
    need = lambda n: lib.mie_moe_prefill_workspace(n, 8, 2, 64, 128, F32)  # noqa: E731
    assert need(0) < 0 or need(0) == INVALID
    assert need(0) < 0
    # Launches take 4096 tokens at a time from one workspace.
    assert need(4096) == need(3 * 4096) and need(4096 + 1) >= need(4096) > need(1) > 0


def test_cpu_layers_keep_the_pytorch_path():
    layer = MoEFeedForward(64, 128, 4, 2).eval()
    x = torch.randn(1, 9, 64)
    with torch.no_grad():
        assert not layer.uses_grouped_prefill(x, decode=False)
        s = layer._expert_storage
        with pytest.raises(RuntimeError):
            fused_moe.prefill(x, layer.router.weight, s["w1"], s["b1"], s["w2"], s["b2"], top_k=2)
        assert torch.equal(layer(x), layer._forward_reference(x))


def test_plain_experts_are_recognised():
    """What decides whether the storages stand in for the experts' modules."""
    layer = MoEFeedForward(16, 32, 3, 2)
    assert layer._experts_are_plain()
    layer.double()
    assert layer._experts_are_plain()
    changes = (
        lambda l: l.experts[0].register_forward_pre_hook(lambda *a: None),
        lambda l: l.experts[2].net[1].register_forward_hook(lambda *a: None),
        lambda l: setattr(l.experts[1].net[2], "bias", torch.nn.Parameter(torch.zeros(16))),
        lambda l: setattr(l.experts[1].net[0].weight, "data", torch.zeros(32, 16)),
        lambda l: l.experts[1].net.__setitem__(1, torch.nn.GELU("tanh")),
        lambda l: l.experts[1].net.__setitem__(1, torch.nn.ReLU()),
        lambda l: l.experts[1].net.append(torch.nn.Identity()),
        lambda l: setattr(l.experts[0], "forward", lambda x: x),
        lambda l: l.experts.__setitem__(0, torch.nn.Identity()),
    )
    for change in changes:
        layer = MoEFeedForward(16, 32, 3, 2)
        change(layer)
        assert not layer._experts_are_plain()


def test_only_plain_inference_is_stood_in_for():
    x = torch.randn(2, 4)
    assert not _native.plain_inference(x)  # gradients on

    class Counting(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with torch.no_grad():
        assert _native.plain_inference(x)
        with torch.device("cpu"):  # a default device changes no operation on x
            assert _native.plain_inference(x)
        with Counting():
            assert not _native.plain_inference(x)
        with torch.autograd.forward_ad.dual_level():
            assert not _native.plain_inference(x)
