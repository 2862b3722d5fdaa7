"""Norm + RoPE + append + attention in one launch against the two launches.

The query rows may differ in the last place (the norm's mean square is summed
in another order), so outputs agree within two roundings of their size: 2^-7
of the largest value for bf16, 2^-10 for f16; the cache rows within one unit.
"""

import numpy as np
import pytest
import torch

from microinfer_amd.layer.hip_paged_attention import decode_plan, hip_paged_decode, hip_qkv_decode
from microinfer_amd.layer.hip_qk_norm_rope import qk_norm_rope_append, rope_tables
from microinfer_amd.workloads import decode_slots, draw_tables
from microinfer_amd.worker.kv_cache import KVCache

pytestmark = pytest.mark.gpu
DEV = "cuda"
D = 128


def _case(contexts, hq, hkv, block_size, dtype, layout, seed=0):
    rng = np.random.default_rng(seed)
    pool = sum(-(-c // block_size) for c in contexts) + 1
    tables = draw_tables(rng, contexts, pool - 1, block_size)
    slots = decode_slots(tables, contexts, block_size)
    gen = torch.Generator(device=DEV).manual_seed(seed)
    caches = []
    for _ in range(2):
        caches.append(KVCache(1, pool, block_size, hkv, D, dtype=dtype, device=DEV,
                              layout=layout))
    fill = torch.randn(2, *caches[0].keys[0].shape, generator=gen, device=DEV).to(dtype)
    for cache in caches:
        cache.keys[0].copy_(fill[0])
        cache.values[0].copy_(fill[1])
    qkv = torch.randn(len(contexts), (hq + 2 * hkv) * D + 16, generator=gen, device=DEV).to(dtype)
    qw = (1 + 0.1 * torch.randn(D, generator=gen, device=DEV)).to(dtype)
    kw = (1 + 0.1 * torch.randn(D, generator=gen, device=DEV)).to(dtype)
    cos, sin = rope_tables(max(contexts) + 3, D, 1e6, device=DEV)
    args = dict(q_weight=qw, k_weight=kw, eps=1e-6, cos_table=cos, sin_table=sin)
    lens = torch.tensor(contexts, dtype=torch.int32, device=DEV)
    return (qkv, torch.tensor(tables, device=DEV), lens,
            torch.tensor(slots, dtype=torch.int32, device=DEV), lens.long() - 1, args,
            [c.layer(0) for c in caches])


def _two_launches(case, hq, hkv, interleaved):
    qkv, tables, lens, slots, positions, args, (cache, _) = case
    q = qk_norm_rope_append(qkv, positions=positions, num_q_heads=hq, num_kv_heads=hkv,
                            head_dim=D, interleaved=interleaved, slot_mapping=slots,
                            key_cache=cache.keys, value_cache=cache.values, **args)
    return hip_paged_decode(q, cache.keys, cache.values, tables, lens)


def _one_launch(case, hq, hkv, interleaved, planned=True):
    qkv, tables, lens, slots, positions, args, (_, cache) = case
    plan = (decode_plan(lens, num_kv_heads=hkv, block_size=cache.block_size,
                        block_table_width=tables.shape[1]) if planned else None)
    return hip_qkv_decode(qkv, cache.keys, cache.values, tables, lens, slots, positions,
                          num_q_heads=hq, interleaved=interleaved, plan=plan, **args)


def _assert_same(case, want, got, dtype):
    unit = 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
    assert float((got.float() - want.float()).abs().max()) <= unit * float(want.abs().max())
    (a, b) = case[-1]
    assert torch.equal(a.values, b.values)
    diff = (a.keys.float() - b.keys.float()).abs()
    assert bool((diff <= unit * a.keys.float().abs() + 1e-6).all())


# One tile, tile and block edges, several partitions, and (40 sequences) the
# narrow launch; groups of 1 to 16 heads over 8 waves.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("contexts,hq,hkv,block_size,layout", [
    ([1], 16, 8, 16, "paired"), ([16, 17, 300, 1500], 16, 8, 16, "paired"),
    ([4000], 32, 8, 16, "head_major"), ([5, 64, 65], 8, 8, 64, "token_major"),
    ([33, 2], 32, 2, 32, "paired"), ([1 + 37 * i for i in range(40)], 16, 8, 16, "paired"),
])
def test_one_launch_is_the_two(contexts, hq, hkv, block_size, layout, interleaved, dtype):
    case = _case(contexts, hq, hkv, block_size, dtype, layout)
    want = _two_launches(case, hq, hkv, interleaved)
    _assert_same(case, want, _one_launch(case, hq, hkv, interleaved), dtype)
    _assert_same(case, want, _one_launch(case, hq, hkv, interleaved, planned=False), dtype)


def test_slots_and_positions_that_are_not_the_end():
    """Skipped, foreign and pad slots and positions past the angle table do
    what the two launches do, as no other row reads those slots."""
    contexts = [40, 33, 50, 1, 20]
    case = list(_case(contexts, 16, 8, 16, torch.bfloat16, "paired"))
    cache = case[-1][0]
    spare = (cache.keys.shape[0] - 1) * 16
    case[3][0] = -1  # not stored: the old row is attended to
    case[3][1] = cache.keys.shape[0] * 16  # outside the cache
    case[3][3] = spare + 5  # a pad row
    case[4][4] = case[5]["cos_table"].shape[0]  # no angles: zero query, nothing stored
    case[4][2] -= 7  # another position: rotated by it
    want = _two_launches(case, 16, 8, False)
    _assert_same(case, want, _one_launch(case, 16, 8, False), torch.bfloat16)


def test_rejects():
    qkv, tables, lens, slots, positions, args, (cache, _) = _case([20, 30], 16, 8, 16,
                                                                  torch.bfloat16, "paired")
    with pytest.raises(ValueError):
        hip_qkv_decode(qkv.float(), cache.keys, cache.values, tables, lens, slots, positions,
                       num_q_heads=16, **args)
    with pytest.raises(ValueError):
        hip_qkv_decode(qkv, cache.keys, cache.values, tables, lens, slots[:1], positions,
                       num_q_heads=16, **args)
    with pytest.raises(ValueError):
        hip_qkv_decode(qkv[:, :512], cache.keys, cache.values, tables, lens, slots, positions,
                       num_q_heads=16, **args)


@pytest.mark.parametrize("seqs,context", [(128, 40), (129, 40), (129, 300)])
def test_model_attends_alike_on_both_routes(seqs, context):
    """Both sides of the line by sequences and table width, through the model's
    own choice, against the two launches."""
    from types import SimpleNamespace

    from microinfer_amd.engine.model import QwenConfig, Qwen3Model
    from microinfer_amd.layer.metadata import AttentionMetadata

    contexts = [1 + (37 * i) % context for i in range(seqs - 1)] + [context]
    case = _case(contexts, 16, 8, 16, torch.bfloat16, "paired")
    qkv, tables, lens, slots, positions, args, (_, cache) = case
    want = _two_launches(case, 16, 8, False)
    metadata = AttentionMetadata.build(is_prefill=False, slot_mapping=slots, context_lens=lens,
                                       block_tables=tables, validate_cache_write=False)
    metadata.slots_at_end = True
    model = Qwen3Model.__new__(Qwen3Model)
    model.config, model.cos, model.sin = QwenConfig(), args["cos_table"], args["sin_table"]
    layer = SimpleNamespace(q_norm=args["q_weight"], k_norm=args["k_weight"])
    got = model._attend(layer, cache, qkv[:, :32 * D].contiguous(), positions, metadata)
    _assert_same(case, want, got.view_as(want), torch.bfloat16)
