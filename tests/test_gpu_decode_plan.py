"""The paged decode's form where only a bound on the lengths is known and where
the lengths are: both against float64, and the block plan's step beside the
per-call path."""

import math

import pytest
import torch

from conftest import print_case
from moe_engine import _native, paged_attention
from moe_engine.model import BlockAllocator, ModelConfig, TransformerMoEBlock
from moe_engine.workloads import make_workload, take_last_tokens

pytestmark = pytest.mark.gpu


def exact(w, k_pool, v_pool):
    out = torch.zeros(w.q.shape, dtype=torch.float64)
    for b, n in enumerate(w.lens):
        ids = w.block_tables[b].long()[: -(-n // w.block_size)]
        k, v = (p[0, ids].transpose(0, 1).reshape(w.q.shape[1], -1, w.q.shape[2])[:, :n].double().cpu()
                for p in (k_pool, v_pool))
        s = (k * w.q[b].double().cpu()[:, None]).sum(-1) / math.sqrt(w.q.shape[2])
        out[b] = (torch.softmax(s, -1)[..., None] * v).sum(1)
    return out


@pytest.mark.parametrize("lens", [[1000], [64], [700, 3, 1000]])
def test_a_bounded_launch_up_to_1024_tokens_takes_no_workspace(lens):
    """mie_paged_decode with device lengths, a bound of 1024 and no workspace.
    Bound on the error: float32 sums of N(0, 1) values, as the decode tests'
    1e-5 for these shapes."""
    w = make_workload(lens, num_heads=12, head_dim=64, block_size=16, dtype=torch.float32, seed=2)
    out = torch.empty_like(w.q)
    print_case("bounded", lens)
    rc = _native.lib().mie_paged_decode(
        w.q.data_ptr(), w.q.stride(0), w.q.stride(1), w.k_pool.data_ptr(), w.v_pool.data_ptr(), w.k_pool.stride(1),
        w.k_pool.stride(2), w.k_pool.shape[1], w.block_tables.data_ptr(), w.block_tables.stride(0),
        w.context_lens.data_ptr(), None, 0, 1024, len(lens), 12, 64, 16, 0.125, out.data_ptr(), out.stride(0),
        out.stride(1), 0, None, 0, 0, 0, _native.stream_of(w.q))
    _native.check(rc, "mie_paged_decode")
    assert (out.double().cpu() - exact(w, w.k_pool, w.v_pool)).abs().max().item() <= 1e-5


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("append", [False, True])
@pytest.mark.parametrize("lens", [[1000], [426], [428, 9], [1000, 1, 700, 1024], [800] * 12])
def test_known_lengths_on_both_sides_of_the_line(lens, append, dtype):
    """8 x 96: float32 rows pass 320 KB at 427 tokens, bfloat16 ones at 854; with
    the append of several sequences the line lies higher."""
    w = make_workload(lens, num_heads=8, head_dim=96, block_size=16, dtype=dtype, seed=6)
    want = exact(w, w.k_pool, w.v_pool)
    pools = w.k_pool.clone(), w.v_pool.clone()
    new = dict(zip(("k_new", "v_new"), take_last_tokens(w))) if append else {}
    print_case("known lengths", lens, append, dtype)
    part, _ = _native.decode_plan_known(len(lens), 8, 96, 16, max(lens), max(lens), append, dtype)
    got = paged_attention.decode_layer(w.q, w.k_pool[0], w.v_pool[0], w.block_tables, context_lens=w.context_lens,
                                       max_context_len=max(lens), context_lens_host=w.lens, **new)
    # bfloat16: the output's rounding, 2^-9 of values up to about 4.
    limit = 1e-5 if dtype == torch.float32 else 1e-2
    assert (got.double().cpu() - want).abs().max().item() <= limit
    assert torch.equal(w.k_pool, pools[0]) and torch.equal(w.v_pool, pools[1])
    # The compiled call takes the same plan.
    if append:
        take_last_tokens(w)
    again = paged_attention.decode_batched(w.q, w.k_pool, w.v_pool, 0, w.block_tables, w.context_lens, max(lens),
                                           context_lens_host=w.lens, **new)
    assert torch.equal(again, got)
    if append:
        take_last_tokens(w)
    forced = paged_attention.decode_batched(w.q, w.k_pool, w.v_pool, 0, w.block_tables, w.context_lens, max(lens),
                                            context_lens_host=w.lens, partition_tokens=part or -1, **new)
    assert torch.equal(forced, got)


@pytest.mark.parametrize("position", [100, 426, 427, 1000])
def test_the_block_plan_splits_known_lengths_and_not_bounds(position):
    """8 x 96 in float32 has no fused attention: the eager step splits rows
    above 320 KB, a step with device counters bounded by the same position
    does not.  Same sums in another order: float32 rounding."""
    torch.manual_seed(1)
    config = ModelConfig(num_layers=1, hidden_dim=768, num_heads=8, num_experts=4, ffn_dim=256)
    block = TransformerMoEBlock(config).to("cuda").eval()
    cache = BlockAllocator(config, 64, 16, "cuda", torch.float32, "direct").new_cache()
    k, v = (torch.randn(1, 8, position, 96, device="cuda") for _ in range(2))
    cache.write(0, 0, k, v)
    x = torch.randn(1, 1, 768, device="cuda")
    print_case("block plan", position)
    with torch.no_grad():
        got = block(x, cache, 0, position).clone()
        plan = block._one_token[2]
        counters = torch.tensor([position, position + 1], dtype=torch.int32, device="cuda")
        rc = _native.lib().mie_block_decode(plan.plan, x.data_ptr(), counters.data_ptr(), position,
                                            _native.stream_of(x))
        _native.check(rc, "mie_block_decode")
        bounded = plan.out.clone()
        block._decode_one_token = lambda *a, **k: None
        want = block(x, cache, 0, position)
    torch.testing.assert_close(got, want, rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(bounded, want, rtol=1e-5, atol=1e-5)
    assert _native.lib().mie_block_plan_launches(plan.plan, position) == 5
