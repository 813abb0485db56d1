"""What decides whether a prompt's attention takes the HIP launches, on the CPU:
the allocator is given a launch record and the device checks answer yes, so
CachedAttention.prompt_supported looks at everything else."""

import pytest
import torch
from torch.nn.utils import parametrize, prune

from moe_engine import _native, paged_attention
from moe_engine.model import BlockAllocator, CachedAttention, ModelConfig, TransformerMoEBlock

DIM, HEADS = 64, 2


class Doubled(torch.nn.Module):
    def forward(self, w):
        return 2 * w


@pytest.fixture
def cache(monkeypatch):
    monkeypatch.setattr(paged_attention, "prefill_supported", lambda *a: True)
    config = ModelConfig(num_layers=1, hidden_dim=DIM, num_heads=HEADS)
    allocator = BlockAllocator(config, 8, 16, "cpu", torch.float32, "auto")
    allocator._launch = (0, 0, 0, _native.DTYPE_CODES[torch.float32])
    return allocator.new_cache()


def pruned(att):
    prune.l1_unstructured(att, "in_proj_weight", 0.5)


def weight_normed(att):
    torch.nn.utils.weight_norm(att, "in_proj_weight")


def parametrized(att):
    parametrize.register_parametrization(att, "in_proj_weight", Doubled())


def parametrized_bias(att):
    parametrize.register_parametrization(att, "in_proj_bias", Doubled())


def plain_weight(att):
    weight = att.in_proj_weight.detach()
    del att.in_proj_weight
    att.in_proj_weight = weight


def wrapped_projection(att):
    inner = att.out_proj
    del att.out_proj
    att.out_proj = lambda x: inner(x)


@pytest.mark.parametrize("change", [pruned, weight_normed, parametrized, parametrized_bias, plain_weight,
                                    wrapped_projection])
def test_projections_that_are_not_registered_parameters_keep_the_pytorch_path(cache, change):
    torch.manual_seed(0)
    att = CachedAttention(DIM, HEADS).eval()
    x = torch.randn(1, 5, DIM)
    with torch.no_grad():
        assert att.prompt_supported(x, cache, 0)
        change(att)
        assert not att.prompt_supported(x, cache, 0)
        # The layer still answers, with what the changed projection computes.
        cache.allocator.on_device = False
        want_qkv = torch.nn.functional.linear(x, att.in_proj_weight, att.in_proj_bias)
        cache.attention_mode = "auto"
        out = att(x, cache, 0, 0)
    q, k, v = (t.view(1, 5, HEADS, -1).transpose(1, 2) for t in want_qkv.chunk(3, dim=-1))
    want = att.out_proj(torch.nn.functional.scaled_dot_product_attention(q, k, v, is_causal=True)
                        .transpose(1, 2).reshape(1, 5, DIM))
    assert torch.equal(out, want)


def test_a_projection_without_bias_is_supported(cache):
    att = CachedAttention(DIM, HEADS).eval()
    att.in_proj_bias = None
    with torch.no_grad():
        assert att.prompt_supported(torch.randn(1, 5, DIM), cache, 0)


@pytest.mark.parametrize("name", ["attn_norm", "moe_norm", "attention", "moe"])
def test_a_part_of_the_block_that_is_no_module_keeps_the_pytorch_path(cache, name):
    block = TransformerMoEBlock(ModelConfig(num_layers=1, hidden_dim=DIM, num_heads=HEADS, num_experts=2)).eval()
    part = getattr(block, name)
    delattr(block, name)
    object.__setattr__(block, name, part)
    with torch.no_grad():
        assert block._prompt(torch.randn(1, 5, DIM), cache, 0) is None
