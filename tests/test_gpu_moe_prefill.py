"""The MoE layer over a prompt (moe_engine.fused_moe.prefill, mie_moe_prefill).

Oracle: the same layer in float64 on the same routing definition (top-k of the
logits, softmax over them, exact GELU), plain torch.  Bounds: a float32 dot
product of n terms accumulated in any order has a relative error of at most
about sqrt(n) * 2^-24 in the 2-norm over many outputs (random signs), so two
chained products of K <= 3072 terms stay below 2 * sqrt(3072) * 2^-24 = 6.6e-6;
in bfloat16 each output passes through at most seven roundings of 2^-9
relative, which add up in the 2-norm to below sqrt(7) * 2^-9 = 5.2e-3, doubled
for roundings upstream of GELU.  Sizes sit at the edges of the tiles (32 and
64 rows, 64 columns, 128 and 256 bytes of K), of a mask word (64 tokens) and
of a launch (4096 tokens).
"""

import pytest
import torch
import torch.nn.functional as F

from conftest import print_case
from moe_engine import fused_moe
from moe_engine.model import MoEFeedForward

pytestmark = pytest.mark.gpu

REL = {torch.float32: 6.6e-6, torch.bfloat16: 1.04e-2}


def moe(dim, hidden, experts, top_k, dtype=torch.float32, seed=0):
    torch.manual_seed(seed)
    return MoEFeedForward(dim, hidden, experts, top_k).to("cuda").to(dtype).eval()


def oracle(layer, x):
    flat = x.double().reshape(-1, x.shape[-1])
    top, ids = torch.topk(F.linear(flat, layer.router.weight.double()), layer.top_k)
    share = torch.softmax(top, -1)
    out = torch.zeros_like(flat)
    for e, expert in enumerate(layer.experts):
        up, _, down = expert.net
        h = F.gelu(F.linear(flat, up.weight.double(), up.bias.double()))
        weight = (share * (ids == e)).sum(-1, keepdim=True)
        out += weight * F.linear(h, down.weight.double(), down.bias.double())
    return out.view(x.shape)


def assert_close(got, want, dtype):
    rel = ((got.double() - want).norm() / want.norm()).item()
    assert rel <= REL[dtype], f"relative error {rel:.2e}"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize(
    "dim,hidden,experts,top_k,tokens",
    [
        (768, 2048, 8, 2, 2), (768, 2048, 8, 2, 63), (768, 2048, 8, 2, 64), (768, 3072, 8, 2, 65),
        (768, 2048, 8, 2, 97), (768, 3072, 8, 2, 1024), (768, 2048, 8, 1, 129), (512, 1024, 16, 4, 300),
        (8, 8, 1, 1, 65), (40, 72, 5, 3, 33), (96, 200, 64, 8, 777), (64, 128, 3, 2, 4097), (2056, 136, 4, 2, 31),
    ],
)
def test_prefill_matches_float64(dim, hidden, experts, top_k, tokens, dtype):
    print_case("moe prefill", dim, hidden, experts, top_k, tokens, dtype)
    layer = moe(dim, hidden, experts, top_k, dtype)
    x = torch.randn(1, tokens, dim, device="cuda").to(dtype)
    with torch.no_grad():
        assert layer.uses_grouped_prefill(x, decode=False)
        got = layer(x)
        assert_close(got, oracle(layer, x), dtype)
        # Rows are summed in one order whatever the workgroups' order.
        assert torch.equal(got, layer(x))


@pytest.mark.parametrize("tokens", [31, 200, 1000])
def test_skewed_routing(tokens):
    """All tokens on the same experts: more rows per expert than the plan's
    average, and experts without a row."""
    layer = moe(64, 128, 8, 2)
    x = torch.randn(1, tokens, 64, device="cuda").abs()
    with torch.no_grad():
        layer.router.weight.copy_(torch.arange(8.0)[:, None].expand(8, 64) * 0.1)
        print_case("skewed", tokens)
        assert_close(layer(x), oracle(layer, x), torch.float32)


def test_batches_views_and_single_tokens():
    layer = moe(64, 128, 4, 2)
    wide = torch.randn(3, 50, 128, device="cuda")
    with torch.no_grad():
        for x in (wide[..., :64], wide[..., 3:67], wide[:, ::2, :64], wide[:1, :1, :64]):
            print_case("view", tuple(x.shape), x.stride())
            assert layer.uses_grouped_prefill(x, decode=False)
            assert_close(layer(x), oracle(layer, x), torch.float32)


def test_special_values_stay_in_their_rows():
    """NaN or infinity in a token reaches that token's row only, as in the
    PyTorch path, and equal logits pick valid experts."""
    layer = moe(64, 128, 4, 2)
    x = torch.randn(1, 70, 64, device="cuda")
    clean = x.clone()
    x[0, 3, 5] = float("nan")
    x[0, 64, 0] = float("inf")
    x[0, 9] = 0.0  # every logit equal
    clean[0, 9] = 0.0
    with torch.no_grad():
        print_case("special values")
        got, want = layer(x), layer(clean)
        assert got[0, 3].isnan().all() and not got[0, 64].isfinite().any()
        rest = [t for t in range(70) if t not in (3, 64)]
        assert torch.equal(got[0, rest], want[0, rest])


def test_applies_only_where_a_library_call_may_stand_in():
    layer = moe(64, 128, 4, 2, torch.bfloat16)
    x = torch.randn(1, 9, 64, device="cuda").bfloat16()
    uses = lambda: layer.uses_grouped_prefill(x, decode=False)  # noqa: E731
    assert not uses()  # gradients on
    with torch.no_grad():
        assert uses()
        assert not layer.uses_grouped_prefill(x.float(), decode=False)
        assert not layer.uses_grouped_prefill(x[:, :1], decode=True)
        with torch.autocast("cuda"):
            assert not uses()
        with torch.autograd.forward_ad.dual_level():
            assert not uses()
        seen = []
        torch.func.vmap(lambda t: seen.append(layer.uses_grouped_prefill(t, decode=False)) or t)(x[None])
        assert seen == [False]
        # bfloat16 experts used to run as modules: a changed one still does.
        handle = layer.experts[1].register_forward_hook(lambda *a: None)
        assert not uses()
        handle.remove()
        assert uses()
        layer.experts[2].net[0].weight = torch.nn.Parameter(torch.zeros(128, 64, device="cuda").bfloat16())
        assert not uses()
        layer._pack_expert_parameters()
        assert uses()
        assert_close(layer(x), oracle(layer, x), torch.bfloat16)
        layer.set_mode("reference")
        assert not uses()
    odd = moe(36, 44, 4, 2, torch.bfloat16)  # rows that are not whole 16-byte vectors
    with torch.no_grad():
        assert not odd.uses_grouped_prefill(torch.randn(1, 9, 36, device="cuda").bfloat16(), decode=False)


def test_captured_prefill_replays_as_eager():
    layer = moe(128, 256, 8, 2)
    x = torch.randn(1, 77, 128, device="cuda")
    with torch.no_grad():
        layer(x)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = layer(x)
        for seed in range(3):
            torch.manual_seed(seed)
            x.copy_(torch.randn(1, 77, 128, device="cuda"))
            want = layer(x)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)


def test_rejects_what_the_kernels_are_not_built_for():
    layer = moe(64, 128, 4, 2)
    s = layer._expert_storage
    weights = (layer.router.weight, s["w1"], s["b1"], s["w2"], s["b2"])
    with torch.no_grad():
        for x in (torch.randn(1, 5, 64), torch.randn(1, 5, 64, device="cuda").double(), torch.randn(1, 5, 60, device="cuda")):
            with pytest.raises(RuntimeError):
                fused_moe.prefill(x, *weights, top_k=2)
        with pytest.raises(RuntimeError):
            fused_moe.prefill(torch.randn(1, 5, 64, device="cuda"), *weights, top_k=5)
