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


@pytest.mark.parametrize("Lq", [37, 64, 150])
@pytest.mark.parametrize("splits", [0, 1, 2, 3])
def test_page_pool_equals_heads_first(gpu, Lq, splits):
    """Requests whose last blocks are different ids, partial where Lq is not a multiple of 64, with NaN
    in every row past their last token: a page pool gives the heads-first cache's output bit for bit."""
    print(f"case: page pool Lq={Lq} splits={splits}", flush=True)
    Hq, Hkv, P = 14, 2, [0, 3, 70, 131]
    B, Qb = len(P), -(-Lq // 64)
    cap = max(P) + Qb
    g = torch.Generator().manual_seed(Lq + splits)
    q = torch.randn((B, Lq, Hq, 128), generator=g).to(torch.bfloat16).to(gpu)
    k, v = (torch.randn((B, Hkv, cap * 64, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    keep = (torch.rand((B, Hkv, cap), generator=g) < 0.6).to(torch.uint8)
    for b, past in enumerate(P):
        k[b, :, 64 * past + Lq:] = float("nan")
        v[b, :, 64 * past + Lq:] = float("nan")
        keep[b, :, past:] = 0
    table, counts = ops.compact_keep_kv(keep.to(gpu), P, Lq, Hq, cap)
    perm = torch.randperm(B * Hkv * cap, generator=g).to(gpu)
    pools = []
    for t in (k, v):
        pool = torch.empty((B * Hkv * cap, 64, 128), dtype=torch.bfloat16, device=gpu)
        pool[perm] = t.view(-1, 64, 128)
        pools.append(pool)
    pages = perm.to(torch.int32).view(B * Hkv, cap)
    scale = 1.0 / math.sqrt(128)
    want, want_lse = ops.attn_fwd(q, ops.KV.heads_first(k), ops.KV.heads_first(v), table, counts, P, scale, cap, Hkv,
                                  with_lse=True, num_splits=splits)
    out, lse = ops.attn_fwd(q, ops.KV.paged(pools[0], pages), ops.KV.paged(pools[1], pages), table, counts, P, scale,
                            cap, Hkv, with_lse=True, num_splits=splits)
    assert torch.equal(out, want) and torch.equal(lse, want_lse)
    k, v = k.nan_to_num(), v.nan_to_num()  # the reference gathers whole blocks (masked for every row)
    torch_reference_check(out, q, k, v, P, table, counts, scale, lse=lse)


def test_dense_decode_of_many_rows_through_a_page_pool(gpu):
    """Decode with more packed rows than its own kernel holds: the block loop over identity lists."""
    print("case: dense decode, 40 packed rows, page pool", flush=True)
    Hq, Hkv, L, lens = 16, 2, 5, [5, 63, 131, 4500]
    cap = -(-max(lens) // 64)
    g = torch.Generator().manual_seed(1)
    q = torch.randn((len(lens), L, Hq, 128), generator=g).to(torch.bfloat16).to(gpu)
    k, v = (torch.randn((len(lens), Hkv, cap * 64, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    for b, n in enumerate(lens):
        k[b, :, n:] = float("nan")
        v[b, :, n:] = float("nan")
    perm = torch.randperm(len(lens) * Hkv * cap, generator=g).to(gpu)
    pools = []
    for t in (k, v):
        pool = torch.empty((len(perm), 64, 128), dtype=torch.bfloat16, device=gpu)
        pool[perm] = t.view(-1, 64, 128)
        pools.append(pool)
    pages = perm.to(torch.int32).view(len(lens) * Hkv, cap)
    scale = 1.0 / math.sqrt(128)
    args = (lens, scale, cap, Hkv)
    want = ops.attn_decode(q, ops.KV.heads_first(k), ops.KV.heads_first(v), *args)
    out = ops.attn_decode(q, ops.KV.paged(pools[0], pages), ops.KV.paged(pools[1], pages), *args)
    assert torch.equal(out, want)
    for b, n in enumerate(lens):
        for h in range(Hq):
            s = (q[b, :, h].float() @ k[b, h * Hkv // Hq, :n].float().T.contiguous()) * scale
            s.masked_fill_(torch.arange(n, device=gpu)[None, :] > torch.arange(n - L, n, device=gpu)[:, None], float("-inf"))
            err = (out[b, :, h].float() - torch.softmax(s, -1) @ v[b, h * Hkv // Hq, :n].float()).abs()
            assert err.max() <= 2e-2 and err.mean() <= 2e-3, (b, h, err.max(), err.mean())


@pytest.mark.parametrize("lens,splits", [
    ([4342, 42073, 460, 1201], 0),            # placement units of one split each
    ([65, 2048, 300] + [200] * 54 + [2048, 2001, 130], 0),  # over 512 splits: whole rows, of 1 and of 3 splits
    ([65, 2048, 300] + [200] * 54 + [2048, 2001, 130], 2),  # whole rows of two splits
])
def test_ragged_decode_placement(gpu, lens, splits):
    """Every way a workgroup of a ragged launch finds its request, KV row and split."""
    print(f"case: ragged decode B={len(lens)} splits={splits}", flush=True)
    B, Hq, Hkv, cap = len(lens), 16, 8, -(-max(lens) // 64)
    g = torch.Generator(device=gpu).manual_seed(B + splits)
    q = torch.randn((B, 1, Hq, 128), generator=g, device=gpu).to(torch.bfloat16)
    k, v = (torch.randn((B, Hkv, cap * 64, 128), generator=g, device=gpu).to(torch.bfloat16) for _ in range(2))
    for b, n in enumerate(lens):
        k[b, :, n:] = float("nan")
        v[b, :, n:] = float("nan")
    scale = 1.0 / math.sqrt(128)
    out = ops.attn_decode(q, ops.KV.heads_first(k), ops.KV.heads_first(v), lens, scale, cap, Hkv, num_splits=splits)
    for b, n in enumerate(lens):
        for h in range(Hkv):
            rows = q[b, 0, 2 * h:2 * h + 2].float()
            s = (rows @ k[b, h, :n].float().T.contiguous()) * scale
            err = (out[b, 0, 2 * h:2 * h + 2].float() - torch.softmax(s, -1) @ v[b, h, :n].float()).abs()
            # the attention tolerances: weights are rounded to bf16, an output is a mean under them
            assert err.max() <= 2e-2 and err.mean() <= 2e-3, (b, h, err.max(), err.mean())


@pytest.mark.parametrize("P", [0, 2])
def test_ids_outside_the_cache_read_its_ends(gpu, P):
    """A table's ids are clamped into the request's blocks, for the causal mask as for the reads."""
    print(f"case: ids outside the cache P={P}", flush=True)
    Hq, Hkv, Lq = 8, 2, 100
    cap = P + 2
    g = torch.Generator().manual_seed(P)
    q = torch.randn((1, Lq, Hq, 128), generator=g).to(torch.bfloat16).to(gpu)
    k, v = (torch.randn((1, Hkv, cap * 64, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    ids = torch.arange(cap, dtype=torch.int32, device=gpu).repeat(Hkv, 1)
    counts = torch.full((Hkv,), cap, dtype=torch.int32, device=gpu)
    args = (counts, [P], 1.0 / math.sqrt(128), cap, Hkv)
    K, V = ops.KV.heads_first(k), ops.KV.heads_first(v)
    want = ops.attn_fwd(q, K, V, ids, *args)
    low = ids.clone()
    low[:, 0] = -5
    assert torch.equal(ops.attn_fwd(q, K, V, low, *args), want)
