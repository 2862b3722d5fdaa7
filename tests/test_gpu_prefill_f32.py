"""float32 varlen attention with head_dim 128 on the float32 MFMA, against the oracle.

The tolerance is that of float32 sums over 128-term dots and a few hundred
keys: 128 * 2^-24 per score in relative terms, values and probabilities of
order one, hence 2e-5.
"""

import math

import numpy as np
import pytest
import torch

from microinfer_amd.layer.hip_paged_attention import hip_paged_prefill
from oracle import dense_causal_attention_f64
from tests.support import as_f32, max_abs, oracle_prefill
from tests.test_gpu_prefill_mfma import D, DEV, _paged_case, _run

pytestmark = pytest.mark.gpu
TOL = 2e-5


# Row tiles are 16 flattened (token, head) rows, key tiles 16 keys; eight
# waves share a tile in launches of few tiles, four in the rest. The block
# size of 8 stays on the vector kernel: the general path, same inputs.
@pytest.mark.parametrize("block_size", [8, 16, 64])
@pytest.mark.parametrize("hq,hkv", [(8, 8), (16, 8), (6, 2), (16, 2)])
@pytest.mark.parametrize("q_lens,prefixes", [
    ([1], [0]), ([3, 1], [13, 200]), ([15, 16, 17, 33, 70], [0, 1, 31, 250, 47]),
])
def test_tile_edges_and_groups(q_lens, prefixes, hq, hkv, block_size):
    if block_size == 8 and hq // hkv not in (1, 2, 8):
        pytest.skip("no vector kernel for this group")
    # Slots past the contexts hold NaN (the vector kernel weighs them by 0).
    case = _paged_case(q_lens, prefixes, hq, hkv, block_size, torch.float32, 3,
                       poison=float("nan") if block_size >= 16 else True)
    q, kc, vc, tables, contexts, cu_q, cu_k = case
    out = _run(q, kc, vc, tables, cu_q, cu_k)
    # The oracle weighs masked slots by 0: give it clean ones.
    expected = oracle_prefill(q, torch.nan_to_num(kc), torch.nan_to_num(vc), tables, contexts,
                              cu_q, 1 / math.sqrt(D))
    assert max_abs(out, expected) <= TOL


def test_more_requests_than_a_wave_scans_at_once():
    q_lens = [1 + 7 * (i % 5) for i in range(70)]
    prefixes = [11 * (i % 9) for i in range(70)]
    q, kc, vc, tables, contexts, cu_q, cu_k = _paged_case(q_lens, prefixes, 16, 8, 16,
                                                          torch.float32, 4)
    out = _run(q, kc, vc, tables, cu_q, cu_k)
    expected = oracle_prefill(q, kc, vc, tables, contexts, cu_q, 1 / math.sqrt(D))
    assert max_abs(out, expected) <= TOL


@pytest.mark.parametrize("length", [1, 16, 37, 300])
def test_contiguous_rows(length):
    # Strided K/V views of a fused row; the arrays end with the last key.
    gen = torch.Generator().manual_seed(length)
    q = torch.randn(length, 4, D, generator=gen)
    kv = torch.randn(length, 4, D, generator=gen)
    fused = kv.to(DEV)
    cu = torch.tensor([0, length], dtype=torch.int32, device=DEV)
    out = hip_paged_prefill(q.to(DEV), fused[:, :2], fused[:, 2:], cu, cu, None,
                            max_seqlen_q=length)
    expected = dense_causal_attention_f64(q.numpy(), kv[:, :2].numpy(), kv[:, 2:].numpy(),
                                          scale=1 / math.sqrt(D))
    assert max_abs(out, expected) <= TOL


def test_invalid_blocks_are_masked_and_nonfinite_values_stay_with_their_rows():
    q, kc, vc, tables, contexts, cu_q, cu_k = _paged_case([40], [30], 16, 8, 16, torch.float32, 5)
    scale = 1 / math.sqrt(D)
    clean = oracle_prefill(q, kc, vc, tables, contexts, cu_q, scale)
    # Position 50 is seen by query rows 20.. only.
    vc[int(tables[0, 50 // 16]), 50 % 16, 3, 7] = float("nan")
    out = as_f32(_run(q, kc, vc, tables, cu_q, cu_k))
    bad = np.zeros_like(clean, dtype=bool)
    bad[20:, 6:8, 7] = True
    assert np.isnan(out[bad]).all()
    assert np.abs(out[~bad] - clean[~bad]).max() <= TOL
    # A table entry outside the pool drops its 16 positions (0-15 here).
    masked = tables.clone()
    masked[0, 0] = kc.shape[0]
    vc = torch.nan_to_num(vc)
    out = as_f32(_run(q, kc, vc, masked, cu_q, cu_k))
    rest = oracle_prefill(q, kc, vc, tables[:, 1:].contiguous(), [c - 16 for c in contexts], cu_q,
                          scale)
    assert np.abs(out - rest).max() <= TOL


def _exact(q, kc, vc, tables, contexts, cu_q):
    """Each request's attention in float64, plain torch."""
    hq, hkv = q.shape[1], kc.shape[2]
    outs = []
    for r, c in enumerate(contexts):
        rows = q[cu_q[r]:cu_q[r + 1]].double()
        n = rows.shape[0]
        ids = tables[r, :-(-c // kc.shape[1])].long()
        k, v = (p[ids].reshape(-1, hkv, D)[:c].double() for p in (kc, vc))
        rows = rows.view(n, hkv, hq // hkv, D).permute(1, 2, 0, 3).reshape(hkv, -1, D)
        s = torch.matmul(rows, k.permute(1, 2, 0).contiguous()) / math.sqrt(D)
        seen = (torch.arange(c, device=DEV)[None] <= torch.arange(c - n, c, device=DEV)[:, None])
        s = s.masked_fill(~seen.repeat(hq // hkv, 1), -math.inf)
        o = torch.matmul(torch.softmax(s, -1), v.permute(1, 0, 2).contiguous())
        outs.append(o.view(hkv, hq // hkv, n, D).permute(2, 0, 1, 3).reshape(n, hq, D))
    return torch.cat(outs)


def test_error_against_64_bits_is_the_vector_kernels():
    """On the same rows: blocks of 8 take the vector kernel. The ratio of the
    two errors is about 1 in the mean; longer summation chains and a second
    rounding of the scaled scores made it 1.06 here."""
    log_ratio = 0.0
    cases = [([200, 90], [100, 0]), ([64] * 4, [0, 30, 300, 7]), ([400], [300]),
             ([300, 25], [0, 9])]
    for seed, (q_lens, prefixes) in enumerate(cases):
        q, kc, vc, tables, contexts, cu_q, cu_k = _paged_case(q_lens, prefixes, 16, 8, 16,
                                                              torch.float32, seed)
        exact = _exact(q, kc, vc, tables, contexts, cu_q)
        halves = torch.stack([2 * tables, 2 * tables + 1], -1).flatten(1)
        narrow = [p.view(-1, 8, *p.shape[2:]) for p in (kc, vc)]
        mfma = _run(q, kc, vc, tables, cu_q, cu_k).double() - exact
        vector = _run(q, *narrow, halves.contiguous(), cu_q, cu_k).double() - exact
        log_ratio += math.log(float(mfma.norm() / vector.norm()))
    assert math.exp(log_ratio / len(cases)) <= 1.03


def test_rows_taken_one_by_one_weigh_scores_of_minus_infinity_by_zero():
    """A NaN in V that only some rows see sends a workgroup's rows through the
    serial path; scores of -inf before any finite one are still weights of 0."""
    q_lens, prefixes = [400], [30]
    q, kc, vc, tables, contexts, cu_q, cu_k = _paged_case(q_lens, prefixes, 16, 8, 16,
                                                          torch.float32, 9)
    q[:, :, 0] = q[:, :, 0].abs() + 0.5
    kc[tables[0, 0].item(), :3, :, 0] = -math.inf  # positions 0-2
    want = _exact(q, kc, vc, tables, contexts, cu_q)
    assert bool(want.isfinite().all())
    vc[tables[0, 50 // 16].item(), 50 % 16, 3, 7] = float("nan")  # seen by rows 20.. only
    got = _run(q, kc, vc, tables, cu_q, cu_k).double()
    bad = torch.zeros_like(got, dtype=torch.bool)
    bad[20:, 6:8, 7] = True
    assert bool(got[bad].isnan().all())
    assert float((got - want)[~bad].abs().max()) <= TOL


@pytest.mark.parametrize("paged", [True, False])
@pytest.mark.parametrize("hq,hkv", [(8, 8), (16, 8), (32, 8), (64, 8), (4, 2), (4, 4)])
def test_few_and_many_rows_agree(hq, hkv, paged):
    """The rows at which the vector kernel hands over to the matrix cores
    (2 to 4 workgroups per CU of rows x KV heads, by the group and the keys):
    the same request, alone and as the last of enough rows."""
    for rows, prefix in ((32, 0), (33, 200), (64, 900), (65, 10), (129, 0)):
        prefix = prefix if paged else 0
        q, kc, vc, tables, contexts, cu_q, cu_k = _paged_case([rows, 400], [prefix, 0], hq, hkv, 16,
                                                              torch.float32, rows)
        want = _exact(q, kc, vc, tables, contexts, cu_q)
        for n, cut in ((1, rows), (2, rows + 400)):
            part = tables[:n, :-(-max(contexts[:n]) // 16)].contiguous()
            if paged:
                got = _run(q[:cut], kc, vc, part, cu_q[:n + 1], cu_k[:n + 1])
            else:
                k, v = (torch.cat([p[tables[r, :-(-c // 16)].long()].reshape(-1, hkv, D)[:c]
                                   for r, c in enumerate(contexts[:n])]) for p in (kc, vc))
                got = _run(q[:cut], k, v, None, cu_q[:n + 1], cu_k[:n + 1])
            assert float((got.double() - want[:cut]).abs().max()) <= TOL
