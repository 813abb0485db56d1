"""The compiled host side of the short calls (moe_engine._host_calls): it takes
the usual form of a call and leaves every other to the Python path, which must
then answer, or raise, as before."""

import sys
import types

import numpy as np
import pytest
import torch

import moe_engine
from conftest import print_case
from moe_engine import _native, kv_ops, paged_attention
from moe_engine.model import BlockAllocator, ModelConfig
from moe_engine.workloads import make_workload


def test_built_and_declines_what_is_not_a_rocm_tensor():
    assert _native.HOST is not None, "moe_engine/_host_calls.so is not built"
    q, pool = torch.zeros(1, 2, 64), torch.zeros(1, 4, 2, 16, 64)
    table, lens = torch.zeros(1, 4, dtype=torch.int32), torch.ones(1, dtype=torch.int32)
    assert _native.HOST.decode(q, pool, pool, 0, table, lens, 1, [1], None, 0, None, None, 0) is None
    assert _native.HOST.gather(pool, pool, 0, table[0], 4, 0) is None
    for args in ((), (None,) * 13, (1,) * 6, ("x",) * 13):
        assert _native.HOST.decode(*args) is None and _native.HOST.gather(*args) is None
    with pytest.raises((TypeError, ValueError)):
        _native.HOST.bind(0, 0, 0, 0)


def test_a_module_built_for_another_abi_is_not_bound(monkeypatch):
    assert _native.HOST.abi_version == _native.ABI_VERSION == _native.lib().mie_abi_version()
    bound = []
    for version in (_native.ABI_VERSION - 1, None, _native.ABI_VERSION):
        stale = types.SimpleNamespace(abi_version=version, __file__="_host_calls.so", bind=lambda *a: bound.append(a))
        monkeypatch.setitem(sys.modules, "moe_engine._host_calls", stale)
        monkeypatch.setattr(moe_engine, "_host_calls", stale, raising=False)
        if version == _native.ABI_VERSION:
            assert _native._open_host() is stale and len(bound) == 1
        else:
            with pytest.warns(RuntimeWarning, match="ABI version"):
                assert _native._open_host() is None
            assert not bound


def calls(w):
    """decode_batched's arguments in forms the compiled call takes and forms
    it leaves; each must give decode_layer's result."""
    q2 = torch.empty(w.q.shape[0], w.q.shape[2], w.q.shape[1], device="cuda", dtype=w.q.dtype).transpose(1, 2)
    q2.copy_(w.q)  # heads innermost
    wide = torch.zeros(*w.q.shape[:2], 2 * w.q.shape[2], device="cuda", dtype=w.q.dtype)
    wide[..., : w.q.shape[2]] = w.q
    tables = torch.zeros(w.block_tables.shape[0], 2 * w.block_tables.shape[1], dtype=torch.int32, device="cuda")
    tables[:, : w.block_tables.shape[1]] = w.block_tables
    return [
        ("plain", w.q, w.block_tables, dict(context_lens_host=w.lens)),
        ("no host lengths", w.q, w.block_tables, {}),
        ("scale", w.q, w.block_tables, dict(scale=0.3, context_lens_host=w.lens)),
        ("integer scale", w.q, w.block_tables, dict(scale=1)),
        ("partitions", w.q, w.block_tables, dict(partition_tokens=256, context_lens_host=w.lens)),
        ("numpy lengths", w.q, w.block_tables, dict(context_lens_host=np.array(w.lens))),
        ("tuple lengths", w.q, w.block_tables, dict(context_lens_host=tuple(w.lens))),
        ("transposed q", q2, w.block_tables, dict(context_lens_host=w.lens)),
        ("strided q", wide[..., : w.q.shape[2]], w.block_tables, dict(context_lens_host=w.lens)),
        ("wide tables", w.q, tables[:, : w.block_tables.shape[1]], dict(context_lens_host=w.lens)),
        ("parameter", torch.nn.Parameter(w.q, requires_grad=False), w.block_tables, dict(context_lens_host=w.lens)),
        ("float32 out", w.q, w.block_tables, dict(out_dtype=torch.float32)),
        ("given out", w.q, w.block_tables, dict(out=torch.empty_like(w.q))),
    ]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_decode_batched_equals_decode_layer(dtype):
    w = make_workload([5, 300, 77, 1000], num_heads=8, head_dim=96, dtype=dtype, layers=2, layer=1, seed=4)
    for name, q, tables, options in calls(w):
        print_case("decode forms", name, dtype)
        options = {k: v.clone() if k == "out" else v for k, v in options.items()}
        got = paged_attention.decode_batched(q, w.k_pool, w.v_pool, 1, tables, w.context_lens, w.max_len, **options)
        want = paged_attention.decode_layer(q, w.k_pool[1], w.v_pool[1], tables, context_lens=w.context_lens,
                                            max_context_len=w.max_len, **options)
        assert got.dtype == want.dtype and got.shape == want.shape and torch.equal(got, want)
    # The last layer by a negative index, as indexing the pools takes it.
    got = paged_attention.decode_batched(w.q, w.k_pool, w.v_pool, -1, w.block_tables, w.context_lens, w.max_len)
    assert torch.equal(got, paged_attention.decode_layer(w.q, w.k_pool[1], w.v_pool[1], w.block_tables,
                                                         context_lens=w.context_lens, max_context_len=w.max_len))


@pytest.mark.gpu
def test_refusals_are_unchanged():
    w = make_workload([5, 30], num_heads=4, head_dim=64, seed=1)
    ok = dict(q=w.q, k_pool=w.k_pool, v_pool=w.v_pool, layer_idx=0, block_tables=w.block_tables,
              context_lens=w.context_lens, max_context_len=w.max_len)
    bad = [
        (dict(q=w.q[0]), ValueError), (dict(q=w.q[:, :2]), ValueError), (dict(q=w.q.float()), ValueError),
        (dict(v_pool=w.v_pool[:, 1:]), ValueError), (dict(layer_idx=1), IndexError),
        (dict(block_tables=w.block_tables.long()), ValueError), (dict(block_tables=w.block_tables[:1]), ValueError),
        (dict(context_lens=w.context_lens[:1]), ValueError), (dict(max_context_len=None), ValueError),
        (dict(q=w.q.cpu()), RuntimeError), (dict(context_lens_host=[1]), ValueError),
        (dict(partition_tokens=100), RuntimeError), (dict(k_new=w.q), ValueError),
        (dict(k_new=w.q, v_new=w.q[:1]), ValueError), (dict(nonsense=1), TypeError),
    ]
    for change, error in bad:
        with pytest.raises(error):
            paged_attention.decode_batched(**{**ok, **change})


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16, torch.float64])
def test_cache_read_equals_the_gather(dtype):
    config = ModelConfig(num_layers=3, hidden_dim=128, num_heads=2)
    cache = BlockAllocator(config, 9, 16, "cuda", dtype, "gather").new_cache()
    k, v = (torch.randn(1, 2, 70, 64, device="cuda").to(dtype) for _ in range(2))
    cache.write(2, 0, k, v)
    for length in (70, 33, 1, 0):
        got = cache.read(2, length)
        assert torch.equal(got[0], k[:, :, :length]) and torch.equal(got[1], v[:, :, :length])
        assert got[0].is_contiguous() and got[0].data_ptr() != got[1].data_ptr() or length == 0
    for layer, length, error in ((3, 4, IndexError), (0, 145, ValueError), (0, -1, ValueError)):
        with pytest.raises(error):
            cache.read(layer, length)
    assert torch.equal(kv_ops.gather(cache.allocator.k_pool, cache.allocator.v_pool, 2, cache.block_table_device, 70)[0], k)
