"""float32 products on the bfloat16 matrix cores (gemm_split.h), through the
prompt MoE and the prompt attention's projections.

Oracle: float64 on the same inputs.  Bound in the 2-norm: the float32 one,
sqrt(K) * 2^-24 per product of K terms, doubled for a chain of two (the split
itself leaves out less than 2^-21 of a product, 2^-24 on average).  Sizes sit
at the edges of its tiles (16 to 64 rows, 64 columns), of a K step (32), of
two steps' loads ahead, and where a row is not whole steps.
"""

import math

import pytest
import torch
import torch.nn.functional as F

from conftest import print_case
from moe_engine.model import BlockAllocator, CachedAttention, ModelConfig, MoEFeedForward

pytestmark = pytest.mark.gpu


def rel(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


def one_expert(dim, hidden, seed=0):
    torch.manual_seed(seed)
    return MoEFeedForward(dim, hidden, 1, 1).to("cuda").eval()


def oracle(layer, x):
    up, _, down = layer.experts[0].net
    h = F.gelu(F.linear(x.double(), up.weight.double(), up.bias.double()))
    return F.linear(h, down.weight.double(), down.bias.double())


@pytest.mark.parametrize("rows", [21, 32, 33, 47, 48, 49, 64, 65, 80, 112, 127])
@pytest.mark.parametrize("dim,hidden", [(4, 8), (28, 36), (32, 64), (36, 68), (64, 132), (100, 96), (128, 260), (768, 2052)])
def test_moe_tile_edges(rows, dim, hidden):
    print_case("split tile", rows, dim, hidden)
    layer = one_expert(dim, hidden)
    x = torch.randn(1, rows, dim, device="cuda")
    with torch.no_grad():
        assert layer.uses_grouped_prefill(x, decode=False)
        got, want = layer(x), oracle(layer, x)
    bound = 2 * math.sqrt(max(dim, hidden)) * 2**-24
    assert rel(got, want) <= max(bound, 2**-21), rel(got, want)


@pytest.mark.parametrize("heads,head_dim,tokens", [(12, 64, 200), (12, 64, 333), (12, 64, 500), (8, 96, 1000), (12, 128, 1024), (24, 128, 1500)])
def test_projections(heads, head_dim, tokens):
    print_case("split projections", heads, head_dim, tokens)
    dim = heads * head_dim
    torch.manual_seed(tokens)
    att = CachedAttention(dim, heads).to("cuda").eval()
    config = ModelConfig(num_layers=1, hidden_dim=dim, num_heads=heads)
    cache = BlockAllocator(config, 100, 16, "cuda", torch.float32, "direct").new_cache()
    x = torch.randn(1, tokens, dim, device="cuda")
    with torch.no_grad():
        att.in_proj_bias.normal_(std=0.1)
        assert att.prompt_supported(x, cache, 0)
        att(x, cache, 0, 0)
        _, k, v = F.linear(x[0].double(), att.in_proj_weight.double(), att.in_proj_bias.double()).chunk(3, -1)
        for got, want in zip(cache.read(0, tokens), (k, v)):
            want = want.view(tokens, heads, head_dim).transpose(0, 1)
            assert rel(got[0], want) <= math.sqrt(dim) * 2**-24


@pytest.mark.parametrize("scale", [1e-30, 1e-18, 1e18, 1e30])
def test_rows_of_any_size_keep_their_precision(scale):
    """Rows far outside the others' range, in A and in W: each as precise as
    alone, and the others bit for bit what they are without them."""
    layer = one_expert(96, 128)
    up, _, down = layer.experts[0].net
    x = torch.randn(1, 100, 96, device="cuda")
    with torch.no_grad():
        up.bias.zero_()
        down.bias.zero_()
        plain = layer(x)
        y = x.clone()
        y[0, 40] *= scale
        got = layer(y)
        print_case("scaled row", scale)
        want = oracle(layer, y[:, 40:41].double())
        # GELU keeps a small row's relative size (x / 2) and a large one's (x or 0).
        assert rel(got[0, 40], want[0, 0]) <= 2**-19
        others = [t for t in range(100) if t != 40]
        assert torch.equal(got[0, others], plain[0, others])
        down.weight[5] *= scale
        scaled = layer(x)
        assert rel(scaled[0, :, 5], oracle(layer, x)[0, :, 5]) <= 2**-19
        columns = [c for c in range(96) if c != 5]
        assert torch.equal(scaled[..., columns], plain[..., columns])


def test_infinities_are_float32s():
    """An infinite value gives infinities where float32 products do, not NaN."""
    att = CachedAttention(768, 12).to("cuda").eval()
    config = ModelConfig(num_layers=1, hidden_dim=768, num_heads=12)
    cache = BlockAllocator(config, 100, 16, "cuda", torch.float32, "direct").new_cache()
    x = torch.randn(1, 400, 768, device="cuda")
    x[0, 399, 17] = float("inf")
    with torch.no_grad():
        print_case("infinite value")
        assert att.prompt_supported(x, cache, 0)
        att(x, cache, 0, 0)
        keys, values = cache.read(0, 400)
        _, k, v = F.linear(x[0, 399].double(), att.in_proj_weight.double()).chunk(3, -1)
        for got, want in ((keys, k), (values, v)):
            assert torch.equal(got[0, :, 399].reshape(-1).double(), want)  # infinities of the same signs
            assert got[0, :, :399].isfinite().all()


@pytest.mark.parametrize("rows", [21, 64, 200])
@pytest.mark.parametrize("dim", [4, 8, 12])
def test_short_sums_are_float32s(rows, dim):
    """Sums of fewer than 16 products keep each product whole.  One value per
    row and column product, the GELU of values above 16 is the value, and W2
    picks one of them: the output is the float32 product, bit for bit."""
    layer = one_expert(dim, 16)
    up, _, down = layer.experts[0].net
    x = torch.zeros(1, rows, dim, device="cuda")
    at = torch.arange(rows, device="cuda") % dim
    value = torch.rand(rows, device="cuda") * 4 + 4
    with torch.no_grad():
        x[0, torch.arange(rows, device="cuda"), at] = value
        up.weight.copy_(torch.rand(16, dim, device="cuda") * 4 + 4)
        up.bias.zero_()
        down.weight.copy_(torch.eye(16, device="cuda")[:dim])
        down.bias.zero_()
        print_case("short sums", rows, dim)
        assert layer.uses_grouped_prefill(x, decode=False)
        got = layer(x)[0]
        assert torch.equal(got, value[:, None] * up.weight[:dim, at].t())
        # A short second product: one hidden value in 4 or 8.
        layer = one_expert(32, dim)
        up, _, down = layer.experts[0].net
        x = torch.zeros(1, rows, 32, device="cuda")
        x[..., 0] = 16 + torch.arange(rows, device="cuda")  # whole numbers: the first product is exact
        up.weight.zero_()
        up.weight[dim - 1, 0] = 1
        up.bias.zero_()
        down.weight.copy_(torch.rand(32, dim, device="cuda") + 1)
        down.bias.zero_()
        got = layer(x)[0]
        assert torch.equal(got, x[0, :, :1] * down.weight[:, dim - 1])
