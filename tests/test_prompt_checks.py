"""What decides whether a prompt's attention takes the HIP launches, on the CPU:
the allocator is given a launch record and the device checks answer yes, so
CachedAttention.prompt_supported looks at everything else."""

import pytest
import torch
from torch.nn.utils import parametrize, prune

from moe_engine import _native, fused_moe, paged_attention
from moe_engine.model import BlockAllocator, CachedAttention, ModelConfig, MoEFeedForward, TransformerMoEBlock

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


class Wrapped(torch.Tensor):
    """A tensor that holds another one and has no memory of its own, as
    quantized and distributed tensors do."""

    @staticmethod
    def __new__(cls, inner):
        return torch.Tensor._make_wrapper_subclass(cls, inner.shape, strides=inner.stride(), dtype=inner.dtype,
                                                   device=inner.device)

    def __init__(self, inner):
        self.inner = inner

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        args, kwargs = torch.utils._pytree.tree_map_only(cls, lambda t: t.inner, (args, kwargs or {}))
        out = func(*args, **kwargs)
        return cls(out) if func is torch.ops.aten.detach.default else out


def replace(module, name, make):
    owner, _, leaf = name.rpartition(".")
    owner = module.get_submodule(owner)
    with torch.no_grad():
        setattr(owner, leaf, torch.nn.Parameter(make(getattr(owner, leaf).detach()), requires_grad=False))


@pytest.mark.parametrize("name", ["in_proj_weight", "in_proj_bias", "out_proj.weight", "out_proj.bias"])
def test_tensors_without_memory_keep_the_pytorch_path(cache, name):
    torch.manual_seed(0)
    att = CachedAttention(DIM, HEADS).eval()
    x = torch.randn(1, 5, DIM)
    with torch.no_grad():
        cache.attention_mode = "gather"
        want = att(x, cache, 0, 0)
        cache.attention_mode = "auto"
        replace(att, name, Wrapped)
        assert att.get_parameter(name).data_ptr() == 0
        assert not att.prompt_supported(x, cache, 0)
        torch.testing.assert_close(att(x, cache, 0, 0), want)


@pytest.mark.parametrize("name", ["attn_norm.weight", "attn_norm.bias", "moe_norm.weight", "moe_norm.bias"])
def test_norms_without_memory_keep_the_pytorch_path(cache, monkeypatch, name):
    monkeypatch.setattr(MoEFeedForward, "uses_grouped_prefill", lambda *a, **k: True)
    monkeypatch.setattr(CachedAttention, "_prompt", lambda self, x, *a, **k: x)
    monkeypatch.setattr(MoEFeedForward, "_forward_grouped", lambda self, x, **k: x)
    block = TransformerMoEBlock(ModelConfig(num_layers=1, hidden_dim=DIM, num_heads=HEADS, num_experts=2)).eval()
    x = torch.randn(1, 5, DIM)
    with torch.no_grad():
        assert block._prompt(x, cache, 0) is x
        replace(block, name, Wrapped)
        assert block._prompt(x, cache, 0) is None


def test_moe_weights_without_memory_keep_the_pytorch_path(monkeypatch):
    monkeypatch.setattr(_native, "is_rocm_device", lambda t: True)
    layer = MoEFeedForward(16, 32, 3, 2).eval()
    x, s = torch.randn(1, 4, 16), layer._expert_storage
    parts = [layer.router.weight, s["w1"], s["b1"], s["w2"], s["b2"]]
    with torch.no_grad():
        assert fused_moe.prefill_supported(x, *parts, 2)
        for i in range(len(parts)):
            changed = [Wrapped(t.detach()) if i == j else t for j, t in enumerate(parts)]
            assert not fused_moe.prefill_supported(x, *changed, 2)
    assert layer._experts_are_plain()

    class Named(torch.Tensor):
        pass

    replace(layer, "experts.1.net.2.bias", lambda t: t.as_subclass(Named))
    assert not layer._experts_are_plain()


@pytest.mark.parametrize("dim,hidden", [(1 << 20, 4), ((1 << 20) + 4, 4), (4, 1 << 20), (4, (1 << 20) + 4)])
def test_supported_widths_are_the_entry_points(monkeypatch, dim, hidden):
    """A width that the launches refuse is declined, not an error."""
    monkeypatch.setattr(_native, "is_rocm_device", lambda t: True)
    parts = [torch.zeros(s) for s in ((1, dim), (1, hidden, dim), (1, hidden), (1, dim, hidden), (1, dim))]
    taken = fused_moe.prefill_supported(torch.zeros(1, 2, dim), *parts, 1)
    assert taken == (max(dim, hidden) <= 1 << 20)
    assert taken == (_native.lib().mie_moe_prefill_workspace(2, 1, 1, dim, hidden, 0) > 0)


@pytest.mark.parametrize("heads,head_dim,dtype,tokens,taken", [
    (12, 64, torch.bfloat16, 1024, True), (12, 64, torch.bfloat16, 1900, True), (12, 64, torch.bfloat16, 2048, False),
    (24, 32, torch.bfloat16, 2048, False), (4, 32, torch.bfloat16, 8192, False), (16, 64, torch.bfloat16, 1536, False),
    (32, 64, torch.bfloat16, 384, True), (32, 64, torch.bfloat16, 640, False), (64, 128, torch.bfloat16, 16, False),
    (12, 64, torch.float32, 16384, True), (12, 64, torch.float32, 32768, False), (32, 64, torch.float32, 2, True),
])
def test_prompts_take_the_launches_where_they_are_faster(cache, heads, head_dim, dtype, tokens, taken):
    dim = heads * head_dim
    config = ModelConfig(num_layers=1, hidden_dim=dim, num_heads=heads)
    allocator = BlockAllocator(config, 1, 16, "cpu", dtype, "auto")
    allocator._launch = cache.allocator._launch
    with torch.device("meta"):
        att = CachedAttention(dim, heads).to(dtype)
    # Parameters of the right shape without their memory filled in.
    att = att.to_empty(device="cpu")
    with torch.no_grad():
        x = torch.empty(1, tokens, dim, dtype=dtype)
        assert att.prompt_supported(x, allocator.new_cache(), 0) is taken


@pytest.mark.parametrize("experts,top_k,dtype,tokens,taken", [
    (1, 1, torch.bfloat16, 39062500, True), (1, 1, torch.bfloat16, 39062501, False),
    (8, 2, torch.bfloat16, 156250000, True), (8, 2, torch.bfloat16, 156250001, False),
    (8, 2, torch.float32, 156250001, True)])
def test_moe_prompts_take_the_launches_where_they_are_faster(monkeypatch, experts, top_k, dtype, tokens, taken):
    """16 x 32 experts: 80e9 operations per expert, 4 T k 16 x 32."""
    monkeypatch.setattr(_native, "is_rocm_device", lambda t: True)
    layer = MoEFeedForward(16, 32, experts, top_k).to(dtype).eval()
    with torch.no_grad():
        x = torch.zeros(1, 1, 16, dtype=dtype).expand(1, tokens, 16)
        assert layer.uses_grouped_prefill(x, decode=False) is taken


def test_experts_with_further_parameters_and_fewer_experts():
    """A parameter a Linear's forward does not read changes nothing; a bias by
    another name, a storage with more experts than the layer has, do."""
    layer = MoEFeedForward(16, 32, 3, 2)
    layer.experts[1].net[2].register_parameter("scale", torch.nn.Parameter(torch.ones(16)))
    assert layer._experts_are_plain()
    layer.experts[2].net[0].register_parameter("scale", torch.nn.Parameter(torch.ones(16)))
    assert layer._experts_are_plain()
    bias = layer.experts[0].net[0].bias
    layer.experts[0].net[0].bias = None
    layer.experts[0].net[0].register_parameter("shift", bias)
    assert not layer._experts_are_plain()
    layer = MoEFeedForward(16, 32, 3, 2)
    del layer.experts[2]
    assert not layer._experts_are_plain()
