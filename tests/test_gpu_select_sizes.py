"""Block logits and row selection at the edges of their dispatch: 16, 32 and 64 query vectors per
workgroup with and without a remainder, rows on both sides of every register count, and
distributions so peaked that most probabilities are subnormal or zero.  Bit for bit."""
from __future__ import annotations

import math

import numpy as np
import oracle
import pytest
import torch

from compactattention_amd import ops

from .util import f32, float_bits_equal, unpack_rowmask

pytestmark = pytest.mark.gpu


def _check(gpu, past, Hkv, G, Qb, spread, seed):
    print(f"case: past={past} Hkv={Hkv} G={G} Qb={Qb} spread={spread}", flush=True)
    B, cap = len(past), max(past) + Qb
    g = torch.Generator().manual_seed(seed)
    qhat = torch.randn((B, Hkv * G, Qb, 128), generator=g) * spread
    khat = torch.randn((B * Hkv, cap, 128), generator=g)
    scale = 1.0 / math.sqrt(128)
    ref = oracle.block_scores(qhat.numpy(), khat.numpy().reshape(B, Hkv, cap, 128), past, scale)
    for kw in (dict(topk=6, sink_blocks=1, local_blocks=2), dict(topk=20, alpha=0.5, topk_all_columns=True)):
        rowmask, scores = ops.score_select(qhat.to(gpu), khat.to(gpu), scale, ops.Rule(**kw), past, Hkv, cap,
                                           with_scores=True)
        assert float_bits_equal(f32(scores), ref)
        assert np.array_equal(unpack_rowmask(rowmask, cap), oracle.select_rows(ref, past, oracle.Rule(**kw)))


@pytest.mark.parametrize("G,Qb", [(1, 1), (5, 3), (16, 1), (9, 2), (16, 2), (11, 3), (16, 4), (13, 5), (5, 16)])
def test_query_vectors_per_workgroup(gpu, G, Qb):
    _check(gpu, [31, 66], 2, G, Qb, 0.3, seed=G * Qb)


@pytest.mark.parametrize("cap", [511, 513, 1024, 1025, 1537, 2304, 2305, 3072, 3073, 4096, 4097])
def test_row_lengths(gpu, cap):
    _check(gpu, [cap - 2], 1, 2, 2, 1.0, seed=cap)


@pytest.mark.parametrize("spread", [9.0, 25.0, 60.0])
@pytest.mark.parametrize("past", [100, 1500])
def test_peaked_rows(gpu, past, spread):
    _check(gpu, [past], 1, 4, 3, spread, seed=past)


@pytest.mark.parametrize("cap", [70, 257, 600, 1500, 2304, 4000, 4200])
def test_nearly_equal_scores_and_many_picks(gpu, cap):
    """Rows whose keys agree in their upper halves, tie, or hold what is no candidate, and more picks than
    a candidate list holds."""
    print(f"case: nearly equal scores cap={cap}", flush=True)
    past, Hkv, G, Qb = [cap - 2, (cap - 2) // 2], 1, 2, 2
    g = torch.Generator().manual_seed(cap)
    x = torch.rand((2, Hkv * G, Qb, cap), generator=g)
    odd = x.clone()
    odd[..., ::7] = float("nan")
    odd[..., 3::11] = float("-inf")
    rows = {"near": 1 + 1e-3 * x, "nearer": 1 + 2e-6 * x, "negative": -1 - 1e-3 * x, "equal": torch.ones_like(x),
            "few": (x * 3).floor(), "late": torch.where(x < 0.9, 0.0, 1 + 1e-4 * x), "odd": 1 + 1e-3 * odd}
    for name, s in rows.items():
        for k in (1, 10, 32, 33, 64, 65, 300):
            for cols in (False, True):
                rule = dict(topk=k, topk_all_columns=cols)
                got = ops.select_scores(s.to(gpu), ops.Rule(**rule), past, Hkv, cap, 64 * Qb)
                want = oracle.select_rows(s.numpy(), past, oracle.Rule(**rule))
                assert np.array_equal(unpack_rowmask(got, cap), want), (name, k, cols)
