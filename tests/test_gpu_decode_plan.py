"""The decode plan's items and their order, against a plain restatement: parts
of one size per sequence in slot order, dispatched largest first. Up to 64
sequences run on the one-wave kernel, more (and forced splits) on the general
one; both follow the same rules."""

import numpy as np
import pytest
import torch

from microinfer_amd.layer.hip_paged_attention import decode_plan, hip_paged_decode, vector_heads

pytestmark = pytest.mark.gpu
TARGET = 192


def _expected(contexts, hkv, block_size, cap=512):
    blocks = [-(-c // block_size) for c in contexts]
    # 64 to cap positions, past 16384 in proportion.
    most = max(cap // block_size, max(blocks) // (16384 // cap))
    least = min(max(max(blocks) // 8, 64 // block_size), most)
    part = max(least, 1, -(-sum(blocks) * hkv // TARGET))
    whole = max((256 if len(contexts) * hkv >= 64 else 160) // block_size,
                min(4, 512 // block_size))
    items, slot = [], 0
    for r in sorted(range(len(blocks)), key=lambda r: (-blocks[r], r)):
        parts = 1 if blocks[r] <= whole else -(-blocks[r] // part)
        for p in range(parts):
            end = blocks[r] if p == parts - 1 else (p + 1) * part
            items.append((end - p * part, slot + p,
                          [r, p * part, end, parts, slot, contexts[r], p, 0]))
        slot += parts
    return [i[2] for i in sorted(items, key=lambda i: (-i[0], i[1]))]


@pytest.mark.parametrize("hkv,block_size", [(8, 16), (1, 16), (2, 64), (8, 256), (4, 8), (8, 1024)])
@pytest.mark.parametrize("contexts", [
    [1], [0, 0], [64, 65, 1], [32768], [40000, 300], [5000, 16, 4999, 0, 16], [100] * 64,
    [161, 160, 130, 400, 1, 2000], [256, 257, 300, 129, 4000] * 3,
    list(range(1, 2049, 32)), [31 * i % 700 for i in range(65)],
])
def test_plan_items_and_order(contexts, hkv, block_size):
    lens = torch.tensor(contexts, dtype=torch.int32, device="cuda")
    width = max(-(-max(contexts) // block_size), 1)
    plan = decode_plan(lens, num_kv_heads=hkv, block_size=block_size, block_table_width=width)
    _assert_items(plan, _expected(contexts, hkv, block_size))
    # The vector kernel's parts are half as long at most.
    plan = decode_plan(lens, num_kv_heads=hkv, block_size=block_size, block_table_width=width,
                       heads=(2 * hkv, 128, torch.float32))
    _assert_items(plan, _expected(contexts, hkv, block_size, cap=256))


def _assert_items(plan, want):
    got = plan.cpu().numpy().view(np.int32).reshape(-1, 8)
    assert got[:len(want)].tolist() == want
    assert (got[len(want):, 0] == -1).all()


@pytest.mark.parametrize("dtype,head_dim,block_size", [
    (torch.float32, 128, 16), (torch.bfloat16, 128, 16), (torch.bfloat16, 64, 16),
    (torch.bfloat16, 128, 8),
])
def test_a_call_without_a_plan_makes_the_shape_s(dtype, head_dim, block_size):
    gen = torch.Generator(device="cuda").manual_seed(0)
    contexts, hkv = [5000, 300, 17], 2
    blocks = [-(-c // block_size) for c in contexts]
    tables = torch.zeros(3, max(blocks), dtype=torch.int32)
    for r, n in enumerate(blocks):
        tables[r, :n] = torch.arange(n) + sum(blocks[:r])
    kc, vc = (torch.randn(sum(blocks), block_size, hkv, head_dim, generator=gen,
                          device="cuda").to(dtype) for _ in range(2))
    q = torch.randn(3, 4, head_dim, generator=gen, device="cuda").to(dtype)
    tables, lens = tables.cuda(), torch.tensor(contexts, dtype=torch.int32, device="cuda")
    heads = vector_heads(q, hkv, block_size)
    assert (heads is None) == (dtype == torch.bfloat16 and head_dim == 128 and block_size == 16)
    plan = decode_plan(lens, num_kv_heads=hkv, block_size=block_size,
                       block_table_width=tables.shape[1], heads=heads)
    own = hip_paged_decode(q, kc, vc, tables, lens)
    assert torch.equal(own, hip_paged_decode(q, kc, vc, tables, lens, plan=plan))


@pytest.mark.parametrize("context", [1000, 4096, 16384, 32768])
def test_parts_cover_as_many_positions_at_every_block_size(context):
    """The launch's workgroups depend on the context, not on how it is cut into
    blocks: no part is longer than the 16-token blocks' by more than a block."""
    longest = {}
    for block_size in (16, 64, 256):
        plan = decode_plan(torch.tensor([context], dtype=torch.int32, device="cuda"),
                           num_kv_heads=8, block_size=block_size,
                           block_table_width=-(-context // block_size))
        items = plan.cpu().numpy().view(np.int32).reshape(-1, 8)
        items = items[items[:, 0] >= 0]
        assert (items[:, 2] - items[:, 1]).sum() == -(-context // block_size)
        longest[block_size] = int((items[:, 2] - items[:, 1]).max()) * block_size
    assert longest[64] <= longest[16] + 64 and longest[256] <= longest[16] + 256
