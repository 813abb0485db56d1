"""Attention over a prompt (moe_engine.paged_attention.prefill,
mie_attn_prefill), alone and as a block's half.

Oracle: float64 torch on the same inputs.  Bounds in the 2-norm: a float32
dot product of n terms has a relative error of about sqrt(n) * 2^-24 at most
(random signs); the chain is two products of dim <= 1024 terms and the
attention's two of at most 1100, so 4 * sqrt(1100) * 2^-24 = 7.9e-6; in
bfloat16 at most four stored values round by 2^-9 on the way (q or k or v,
the attention's output, the projection's, the residual sum), and rounded
scores move the softmax by as much again: 8 * 2^-9 / 2 = 7.8e-3.  Lengths sit
at the edges of the attention's tiles (16 queries, 32 keys per wave, 128 per
workgroup step), of the projections' forms (12 x 64: QKV leaves the direct tiles
after 32 tokens, the output projection takes larger direct tiles from 65 and
leaves them after 160) and of blocks.
"""

import math

import pytest
import torch
import torch.nn.functional as F

from conftest import print_case
from moe_engine import paged_attention
from moe_engine.model import CachedAttention, Model, ModelConfig, TransformerMoEBlock

pytestmark = pytest.mark.gpu

REL = {torch.float32: 7.9e-6, torch.bfloat16: 7.8e-3}


def oracle(att, x, norm=None):
    x = x[0].double()
    y = x if norm is None else F.layer_norm(x, x.shape[-1:], norm.weight.double(),
                                            None if norm.bias is None else norm.bias.double(), norm.eps)
    n, heads = x.shape[0], att.num_heads
    bias = None if att.in_proj_bias is None else att.in_proj_bias.double()
    q, k, v = (t.view(n, heads, -1).transpose(0, 1) for t in
               F.linear(y, att.in_proj_weight.double(), bias).chunk(3, -1))
    scores = q @ k.transpose(1, 2).contiguous() / math.sqrt(q.shape[-1])
    scores = scores.masked_fill(torch.ones(n, n, dtype=torch.bool, device=x.device).triu(1), -math.inf)
    a = (torch.softmax(scores, -1) @ v.contiguous()).transpose(0, 1).reshape(n, -1)
    out = F.linear(a, att.out_proj.weight.double(), None if att.out_proj.bias is None else att.out_proj.bias.double())
    return (out if norm is None else out + x)[None], k, v


def rel(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


def allocator(heads, head_dim, layers, blocks, block_size, dtype, mode="direct"):
    from moe_engine.model import BlockAllocator

    config = ModelConfig(num_layers=layers, hidden_dim=heads * head_dim, num_heads=heads)
    return BlockAllocator(config, blocks, block_size, "cuda", dtype, mode)


def attention(dim, heads, dtype, seed=0):
    torch.manual_seed(seed)
    att = CachedAttention(dim, heads).to("cuda").to(dtype).eval()
    with torch.no_grad():
        att.in_proj_bias.normal_(std=0.1)
    return att


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize(
    "heads,head_dim,block_size,tokens",
    [
        (12, 64, 16, 1), (12, 64, 16, 15), (12, 64, 16, 17), (12, 64, 16, 62), (12, 64, 16, 129),
        (12, 64, 16, 256), (12, 64, 16, 257), (12, 64, 16, 1024), (8, 96, 16, 33), (8, 96, 16, 300),
        (2, 32, 7, 100), (3, 32, 16, 513), (4, 128, 32, 65), (8, 128, 32, 1000), (1, 64, 1, 31),
        (12, 64, 16, 32), (12, 64, 16, 33), (12, 64, 16, 64), (12, 64, 16, 65), (12, 64, 16, 160), (12, 64, 16, 161),
    ],
)
def test_prompt_matches_float64(heads, head_dim, block_size, tokens, dtype):
    print_case("prompt attention", heads, head_dim, block_size, tokens, dtype)
    dim = heads * head_dim
    att = attention(dim, heads, dtype)
    blocks = -(-tokens // block_size) + 2
    alloc = allocator(heads, head_dim, 2, blocks, block_size, dtype)
    # No order in the table; a cache of another sequence keeps its block.
    other = alloc.new_cache()
    other._reserve(1)
    alloc.free_blocks = [alloc.free_blocks[i] for i in torch.randperm(len(alloc.free_blocks)).tolist()]
    cache = alloc.new_cache()
    x = torch.randn(1, tokens, dim, device="cuda").to(dtype)
    with torch.no_grad():
        assert att.prompt_supported(x, cache, 1)
        got = att(x, cache, 1, 0)
        want, k, v = oracle(att, x)
        assert rel(got, want) <= REL[dtype], rel(got, want)
        keys, values = cache.read(1, tokens)
        assert rel(keys[0], k) <= REL[dtype] and rel(values[0], v) <= REL[dtype]
    # Layer 0, the other sequence's block and the slots past the prompt stay zero.
    used = torch.zeros(blocks, block_size, dtype=torch.bool)
    t = torch.arange(tokens)
    used[torch.tensor(cache.block_table)[t // block_size], t % block_size] = True
    for pool in (alloc.k_pool, alloc.v_pool):
        assert not pool[0].any()
        assert not pool[1].transpose(1, 2)[~used.to("cuda")].any()


def test_heavy_keys():
    """Scores of hundreds: the running maximum moves late."""
    att = attention(128, 2, torch.float32)
    cache = allocator(2, 64, 1, 32, 16, torch.float32).new_cache()
    x = torch.randn(1, 300, 128, device="cuda")
    x[:, 200:210] *= 30
    with torch.no_grad():
        print_case("heavy keys")
        # Products of large terms: the error is relative to the scores.
        assert rel(att(x, cache, 0, 0), oracle(att, x)[0]) <= 1e-4


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens", [1, 31, 200])
def test_block_prompt_matches_its_modules(tokens, dtype):
    """The block's launches against its own modules one by one."""
    config = ModelConfig(max_seq_length=256, num_layers=1, hidden_dim=128, num_heads=2, num_experts=4, top_k=2,
                         ffn_dim=256)
    torch.manual_seed(1)
    block = TransformerMoEBlock(config).to("cuda").to(dtype).eval()
    x = torch.randn(1, tokens, 128, device="cuda").to(dtype)
    new = lambda: allocator(2, 64, 1, 16, 16, dtype).new_cache()  # noqa: E731
    with torch.no_grad():
        print_case("block prompt", tokens, dtype)
        assert block._prompt(x, new(), 0) is not None
        fused_cache, plain_cache = new(), new()
        got = block(x, fused_cache, 0, 0)
        handle = block.attn_norm.register_forward_hook(lambda *a: None)  # keeps the modules
        assert block._prompt(x, new(), 0) is None
        want = block(x, plain_cache, 0, 0)
        handle.remove()
    bound = {torch.float32: 1e-5, torch.bfloat16: 2e-2}[dtype]  # two halves of the bounds above
    assert rel(got, want.double()) <= bound
    assert rel(fused_cache.allocator.k_pool, plain_cache.allocator.k_pool.double()) <= bound


def test_falls_back_where_a_library_call_may_not_stand_in():
    att = attention(128, 2, torch.float32)
    alloc = allocator(2, 64, 1, 8, 16, torch.float32)
    cache = alloc.new_cache()
    x = torch.randn(1, 20, 128, device="cuda")
    assert not att.prompt_supported(x, cache, 0)  # gradients on
    out = att(x, cache, 0, 0)
    assert out.requires_grad
    with torch.no_grad():
        assert att.prompt_supported(x, cache, 0)
        assert not att.prompt_supported(x.bfloat16(), cache, 0)
        assert not att.prompt_supported(x, cache, 1)
        assert not att.prompt_supported(x.expand(2, 20, 128), cache, 0)
        assert not att.prompt_supported(x, allocator(4, 32, 1, 8, 16, torch.float32).new_cache(), 0)
        assert not att.prompt_supported(x, allocator(2, 64, 1, 8, 16, torch.float32, "gather").new_cache(), 0)
        with torch.autocast("cuda"):
            assert not att.prompt_supported(x, cache, 0)
        handle = att.out_proj.register_forward_hook(lambda *a: None)
        assert not att.prompt_supported(x, cache, 0)
        handle.remove()
        # Views and transposed inputs are what they were.
        wide = torch.randn(1, 256, 20, device="cuda")
        view = wide[:, :128].transpose(1, 2)
        assert rel(att(view, cache, 0, 0), oracle(att, view)[0]) <= REL[torch.float32]
        full = allocator(2, 64, 1, 1, 16, torch.float32).new_cache()
        with pytest.raises(RuntimeError, match="no free KV cache blocks"):
            att(x, full, 0, 0)
        assert full.block_table == [] and not full.allocator.k_pool.any()


def test_model_prompt_then_decode_matches_contiguous_cache():
    torch.manual_seed(0)
    model = Model(ModelConfig(max_seq_length=128, vocab_size=512, num_layers=3, hidden_dim=128, num_heads=2,
                              num_experts=4, top_k=2)).to("cuda").eval()
    ids = torch.randint(0, 512, (70,), device="cuda")
    print_case("model prompt")
    want = model.generate(ids, max_new_tokens=12, temperature=0)
    cache = model.new_block_allocator(num_blocks=8, block_size=16, attention_mode="direct").new_cache()
    assert torch.equal(model.generate(ids, max_new_tokens=12, temperature=0, cache=cache), want)


def test_unbuilt_heads_keep_the_pytorch_path():
    assert not paged_attention.prefill_supported(4, 48, torch.float32)
    assert not paged_attention.prefill_supported(4, 64, torch.float64)
    att = attention(96, 2, torch.float32)  # head_dim 48: not built
    cache = allocator(2, 48, 1, 8, 16, torch.float32, "auto").new_cache()
    x = torch.randn(1, 20, 96, device="cuda")
    with torch.no_grad():
        assert not att.prompt_supported(x, cache, 0)
        assert rel(att(x, cache, 0, 0), oracle(att, x)[0]) <= REL[torch.float32]
