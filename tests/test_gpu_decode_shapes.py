"""Decode attention at the edges of its launch shapes: eight waves a workgroup up to 256 workgroups, four beyond; one split or
several; splits that are empty; more splits than the second pass reads side by side."""
import math

import numpy as np
import pytest
import torch


import oracle
from oracle import libtorch_path as lt
from tests.util import bits, from_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,L,D,splits", [
    (32, 8, 8, 40, 128, 1), (33, 8, 8, 40, 128, 1),            # 256 and 264 workgroups, one split
    (4, 16, 16, 130, 128, 4), (5, 16, 16, 130, 128, 4),        # 256 and 320, four splits
    (1, 4, 2, 2100, 128, 64), (1, 2, 1, 2100, 64, 64),         # the most splits
    (1, 2, 2, 600, 128, 33), (1, 2, 2, 600, 64, 17),           # one more than a pass takes at once / side by side; empty splits
    (1, 16, 1, 385, 128, 0), (3, 8, 8, 384, 64, 0), (17, 8, 8, 400, 64, 0),
])
@pytest.mark.parametrize("lens", [False, True])
def test_decode_launch_shapes(B, Hq, Hkv, L, D, splits, lens):
    import tyr_amd as gpu
    q, = lt.make_inputs(40 + L, (B, Hq, 1, D))
    k, v = lt.make_inputs(41 + L, (B, Hkv, L, D), (B, Hkv, L, D))
    n = [L - (i * 7919) % L if lens else L for i in range(B)]
    kv_lens = torch.tensor(n, dtype=torch.int32, device="cuda") if lens else None
    sc = 1 / math.sqrt(D)
    o, lse = gpu.gqa_decode(q.cuda(), k.cuda(), v.cuda(), scale=sc, num_splits=splits, kv_lens=kv_lens)
    for b in sorted({0, B // 2, B - 1}):
        kb, vb = k[b:b + 1, :, :n[b]].contiguous(), v[b:b + 1, :, :n[b]].contiguous()
        want_o, want_lse = oracle.gqa_decode(bits(q[b:b + 1]), bits(kb), bits(vb), sc, 1)
        assert float((o[b:b + 1].cpu().float() - from_bits(want_o).float()).abs().max()) <= 8e-3, (b, n[b])
        assert float(np.abs(lse[b:b + 1].cpu().numpy() - np.asarray(want_lse)).max()) <= 1e-3, (b, n[b])


@pytest.mark.parametrize("Hq,Hkv,L,D,splits", [(4, 2, 1056, 128, 33), (2, 1, 2048, 128, 64), (4, 1, 2017, 64, 64), (8, 8, 1500, 128, 23),
                                               (4, 4, 33, 128, 4), (2, 2, 20, 64, 4)])
@pytest.mark.parametrize("window", [0, 19, 1000])
def test_more_splits_than_chunks_with_rows(Hq, Hkv, L, D, splits, window):
    """Counts whose chunks, rounded up to whole steps, are fewer than asked for, down to one; and 33 and 64 that all hold rows."""
    import tyr_amd as gpu
    q, = lt.make_inputs(60 + L, (1, Hq, 1, D))
    k, v = lt.make_inputs(61 + L, (1, Hkv, L, D), (1, Hkv, L, D))
    sc = 1 / math.sqrt(D)
    o, lse = gpu.gqa_decode(q.cuda(), k.cuda(), v.cuda(), scale=sc, num_splits=splits, window=window)
    lo = max(0, L - window) if window else 0
    want_o, want_lse = oracle.gqa_decode(bits(q), bits(k[:, :, lo:].contiguous()), bits(v[:, :, lo:].contiguous()), sc, 1)
    assert float((o.cpu().float() - from_bits(want_o).float()).abs().max()) <= 8e-3
    assert float(np.abs(lse.cpu().numpy() - np.asarray(want_lse)).max()) <= 1e-3
