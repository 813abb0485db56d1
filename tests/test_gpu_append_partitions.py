"""The append fused into the partition form of the paged decode: against the
append launch followed by the plain decode, on the sequence lengths where a
partition ends, begins with the new token alone, or is the only one.

The new token's score and value come from registers instead of the pool, with
the same arithmetic; it joins its wave's softmax state last instead of in its
tile, so outputs may differ by float32 rounding of the merge: 2^-22 of the
largest value times a few operations, below 4e-6 for N(0, 1) values.  Pools
must be equal bit for bit.
"""

import pytest
import torch

from conftest import print_case
from moe_engine import kv_ops, paged_attention
from moe_engine.workloads import make_workload, take_last_tokens

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,head_dim,block_size", [(12, 64, 16), (8, 96, 16), (3, 128, 32), (5, 64, 12), (2, 4, 8)])
def test_fused_append_equals_append_then_decode(heads, head_dim, block_size, dtype):
    # 256-token partitions whatever the tile (head_dim 4 has the largest).
    lens = [1, 2, 31, 32, 33, 255, 256, 257, 258, 512, 513, 1000, 0]
    part = 1024 if head_dim == 4 else 256
    w = make_workload(lens, num_heads=heads, head_dim=head_dim, block_size=block_size, dtype=dtype, seed=3)
    k_new, v_new = take_last_tokens(w)
    pools = [t.clone() for t in (w.k_pool, w.v_pool)]
    print_case("append in partitions", heads, head_dim, block_size, dtype)
    got = paged_attention.decode_batched(
        w.q, w.k_pool, w.v_pool, 0, w.block_tables, w.context_lens, w.max_len, partition_tokens=part,
        context_lens_host=w.lens, k_new=k_new, v_new=v_new, out_dtype=torch.float32)
    kv_ops.append(*pools, 0, k_new[:, :, None], v_new[:, :, None], w.block_tables,
                  positions=(w.context_lens - 1).contiguous())
    want = paged_attention.decode_batched(
        w.q, *pools, 0, w.block_tables, w.context_lens, w.max_len, partition_tokens=part, context_lens_host=w.lens,
        out_dtype=torch.float32)
    assert torch.equal(w.k_pool, pools[0]) and torch.equal(w.v_pool, pools[1])
    assert (got - want).abs().max().item() <= 4e-6
    # Each sequence alone (the fused form), from pools without the new rows.
    for b, n in enumerate(lens):
        w1 = make_workload(lens, num_heads=heads, head_dim=head_dim, block_size=block_size, dtype=dtype, seed=3)
        take_last_tokens(w1)
        alone = paged_attention.decode_batched(
            w1.q[b : b + 1], w1.k_pool, w1.v_pool, 0, w1.block_tables[b : b + 1], w1.context_lens[b : b + 1], max(n, 1),
            partition_tokens=part, context_lens_host=[n], k_new=k_new[b : b + 1], v_new=v_new[b : b + 1],
            out_dtype=torch.float32)
        assert (alone[0] - want[b]).abs().max().item() <= 4e-6
        if n > 0:
            at = w.block_tables[b, (n - 1) // block_size], (n - 1) % block_size
            for mine, theirs in ((w1.k_pool, pools[0]), (w1.v_pool, pools[1])):
                assert torch.equal(mine[0, at[0], :, at[1]], theirs[0, at[0], :, at[1]])
    # A launch bound instead of the exact list, and a bad block id for one sequence.
    again = paged_attention.decode_batched(
        w.q, w.k_pool, w.v_pool, 0, w.block_tables, w.context_lens, w.max_len, partition_tokens=part, k_new=k_new,
        v_new=v_new, out_dtype=torch.float32)
    assert torch.equal(again, got)
    tables = w.block_tables.clone()
    last = (w.lens[8] - 1) // block_size
    tables[8, last] = -1
    before = w.k_pool.clone()
    bad = paged_attention.decode_batched(
        w.q, w.k_pool, w.v_pool, 0, tables, w.context_lens, w.max_len, partition_tokens=part, context_lens_host=w.lens,
        k_new=k_new, v_new=v_new, out_dtype=torch.float32)
    assert bad[8].isnan().all() and torch.equal(w.k_pool, before)
    rest = [b for b in range(len(lens)) if b != 8]
    assert torch.equal(bad[rest], got[rest])


def test_rows_of_one_sequence_see_each_others_tokens():
    """Three rows share one block table at lengths n, n + 1, n + 2: each
    attends to the tokens the shorter ones append in the same call."""
    w = make_workload([700], num_heads=12, head_dim=64, block_size=16, dtype=torch.float32, seed=5)
    lens = [698, 699, 700]
    tables = w.block_tables.expand(3, -1).contiguous()
    q, k_new, v_new = (torch.randn(3, 12, 64, device="cuda") for _ in range(3))
    context = torch.tensor(lens, dtype=torch.int32, device="cuda")
    print_case("shared table")
    got = paged_attention.decode_batched(q, w.k_pool, w.v_pool, 0, tables, context, 700, partition_tokens=256,
                                         context_lens_host=lens, k_new=k_new, v_new=v_new)
    want = paged_attention.decode_batched(q, w.k_pool, w.v_pool, 0, tables, context, 700, partition_tokens=256,
                                          context_lens_host=lens)
    assert torch.equal(got, want)
    ids = tables[0].long()
    for pool, new in ((w.k_pool, k_new), (w.v_pool, v_new)):
        rows = pool[0, ids].transpose(0, 1).reshape(12, -1, 64)[:, 697:700]
        assert torch.equal(rows, new.transpose(0, 1))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lens", [[698, 699, 700], [15, 17, 16], [700, 700]])
def test_rows_that_share_their_last_blocks_in_both_documented_ways(lens, dtype):
    """Rows of one sequence at several lengths: appended by their own launch and
    then decoded in every form, and by the fused entry with partitions
    requested.  Oracle: float64 attention over the pools with every row's token
    in (for two rows of one length, the same token)."""
    w = make_workload([max(lens)], num_heads=12, head_dim=64, block_size=16, dtype=dtype, seed=5)
    rows = len(lens)
    tables = w.block_tables.expand(rows, -1).contiguous()
    q, k_new, v_new = (torch.randn(rows, 12, 64, device="cuda").to(dtype) for _ in range(3))
    if len(set(lens)) == 1:
        k_new, v_new = (t[:1].expand(rows, -1, -1).contiguous() for t in (k_new, v_new))
    context = torch.tensor(lens, dtype=torch.int32, device="cuda")
    pools = [t.clone() for t in (w.k_pool, w.v_pool)]
    print_case("shared last block", lens, dtype)
    kv_ops.append(*pools, 0, k_new[:, :, None], v_new[:, :, None], tables, positions=context - 1)
    k, v = (p[0, tables[0].long()].transpose(0, 1).reshape(12, -1, 64).double() for p in pools)
    want = torch.stack([
        (torch.softmax((k[:, :n] * q[b].double()[:, None]).sum(-1) / 8, -1)[..., None] * v[:, :n]).sum(1)
        for b, n in enumerate(lens)])
    # float32 sums of N(0, 1) values, as the decode tests' 1e-5; bfloat16 adds the output's rounding, 2^-9 of
    # values below 4.
    limit = 1e-5 if dtype == torch.float32 else 1e-2
    for part in (0, -1, 256):
        got = paged_attention.decode_batched(q, *pools, 0, tables, context, max(lens), partition_tokens=part,
                                             context_lens_host=lens)
        assert (got.double() - want).abs().max().item() <= limit
    got = paged_attention.decode_batched(q, w.k_pool, w.v_pool, 0, tables, context, max(lens), partition_tokens=256,
                                         context_lens_host=lens, k_new=k_new, v_new=v_new)
    assert (got.double() - want).abs().max().item() <= limit
    assert torch.equal(w.k_pool, pools[0]) and torch.equal(w.v_pool, pools[1])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16, torch.float64])
@pytest.mark.parametrize("heads,head_dim,block_size,length", [(12, 64, 16, 8192), (12, 64, 16, 4097), (40, 24, 7, 3001),
                                                              (12, 64, 16, 1)])
def test_gather_with_several_vectors_per_thread(heads, head_dim, block_size, length, dtype):
    """Lengths on both sides of the switch to four vectors per thread, with a
    tail, against the indexed rebuild; rows of a bad block id stay unwritten."""
    blocks = -(-length // block_size) + 3
    pools = [torch.randn(1, blocks, heads, block_size, head_dim, device="cuda").to(dtype) for _ in range(2)]
    table = torch.randperm(blocks)[: -(-length // block_size)].to(torch.int32).to("cuda")
    print_case("gather", heads, head_dim, block_size, length, dtype)
    want = [p[0, table.long()].transpose(0, 1).reshape(heads, -1, head_dim)[:, :length] for p in pools]
    got = kv_ops.gather(*pools, 0, table, length)
    assert all(torch.equal(g[0], w) for g, w in zip(got, want))
    table[-1] = blocks
    out = [torch.full((1, heads, length, head_dim), 7, dtype=dtype, device="cuda") for _ in range(2)]
    kv_ops.gather(*pools, 0, table, length, *out)
    start = (len(table) - 1) * block_size
    for o, w in zip(out, want):
        assert torch.equal(o[0, :, :start], w[:, :start]) and (o[0, :, start:] == 7).all()
