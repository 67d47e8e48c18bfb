"""The attention kernel's block loop at every list length where its parts change: lists shorter
than the load rings, lists that leave 0 to 3 blocks after the four-block rounds, and lists that
cross the 64 entries read at a time."""
from __future__ import annotations

import math

import pytest
import torch

from compactattention_amd import ops

from .util import torch_reference_check

pytestmark = pytest.mark.gpu


def _case(gpu, kept, Lq, Hq, Hkv, layout, splits):
    """One request of max(kept) + 5 past blocks whose KV row h keeps kept[h] of them."""
    print(f"case: kept={kept} Lq={Lq} layout={layout} splits={splits}", flush=True)
    g = torch.Generator().manual_seed(sum(kept) + Lq)
    P = max(kept) + 5
    Qb = -(-Lq // 64)
    cap = P + Qb
    q = torch.randn((1, Lq, Hq, 128), generator=g).to(torch.bfloat16).to(gpu)
    k, v = (torch.randn((1, Hkv, cap * 64, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    live = 64 * P + Lq
    k[:, :, live:] = float("nan")  # rows past the request's last token are never used
    v[:, :, live:] = float("nan")
    keep = torch.zeros((1, Hkv, cap), dtype=torch.uint8)
    for h, n in enumerate(kept):
        keep[0, h, torch.randperm(P, generator=g)[:n]] = 1
    table, counts = ops.compact_keep_kv(keep.to(gpu), [P], Lq, Hq, cap)
    assert counts.tolist() == [n + Qb for n in kept]
    if layout == "heads_first":
        K, V = ops.KV.heads_first(k), ops.KV.heads_first(v)
    elif layout == "seq_first":
        K, V = ops.KV.seq_first(k.transpose(1, 2).contiguous()), ops.KV.seq_first(v.transpose(1, 2).contiguous())
    else:
        perm = torch.randperm(Hkv * cap, generator=g)
        pools = []
        for t in (k, v):
            pool = torch.empty((Hkv * cap, 64, 128), dtype=torch.bfloat16, device=gpu)
            pool[perm.to(gpu)] = t.view(Hkv * cap, 64, 128)
            pools.append(pool)
        pt = perm.to(torch.int32).view(Hkv, cap).to(gpu)
        K, V = ops.KV.paged(pools[0], pt), ops.KV.paged(pools[1], pt)
    scale = 1.0 / math.sqrt(128)
    out, lse = ops.attn_fwd(q, K, V, table, counts, [P], scale, cap, Hkv, with_lse=True, num_splits=splits)
    # the tolerances of the attention output and of log-sum-exps over bf16-rounded weights
    torch_reference_check(out, q, k[:, :, :live], v[:, :, :live].contiguous(), [P], table, counts, scale, lse=lse) \
        if Lq % 64 == 0 else _check_partial(out, q, k, v, P, live, table, counts, scale, lse)


def _check_partial(out, q, k, v, P, live, table, counts, scale, lse):
    # the reference gathers whole blocks: give it zeros past the last token (masked for every row)
    k, v = k.clone(), v.clone()
    k[:, :, live:] = 0
    v[:, :, live:] = 0
    torch_reference_check(out, q, k, v, [P], table, counts, scale, lse=lse)


@pytest.mark.parametrize("layout", ["heads_first", "seq_first", "paged"])
def test_list_lengths(gpu, layout):
    for first in (0, 4, 8, 61, 65, 125):
        _case(gpu, [first, first + 1, first + 2, first + 3], 64, 16, 4, layout, 1)


@pytest.mark.parametrize("layout", ["heads_first", "seq_first", "paged"])
def test_list_lengths_partial_block_and_splits(gpu, layout):
    _case(gpu, [3, 66], 37, 14, 2, layout, 1)
    _case(gpu, [130, 7], 150, 14, 2, layout, 3)
    _case(gpu, [259, 200], 64, 8, 2, layout, 2)
