"""Dense decode on both sides of the size from which K and V are loaded without staying in the
last-level cache (320 MB of K and V: 81920 tokens of 8 heads)."""
from __future__ import annotations

import math

import pytest
import torch

from compactattention_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["heads_first", "seq_first", "paged"])
@pytest.mark.parametrize("lens", [[80001, 1918], [80001, 1919], [45000, 40000, 77]])
def test_decode_around_the_cache_size(gpu, lens, layout):
    print(f"case: decode lens={lens} layout={layout}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(sum(lens))
    B, Hq, Hkv, cap = len(lens), 32, 8, (max(lens) + 63) // 64
    q = torch.randn((B, 1, Hq, 128), generator=g, device=gpu).to(torch.bfloat16)
    k, v = (torch.randn((B, Hkv, cap * 64, 128), generator=g, device=gpu).to(torch.bfloat16) for _ in range(2))
    for b, n in enumerate(lens):  # rows past the request's last token are never used
        k[b, :, n:] = float("nan")
        v[b, :, n:] = float("nan")
    if layout == "heads_first":
        K, V = ops.KV.heads_first(k), ops.KV.heads_first(v)
    elif layout == "seq_first":
        K, V = (ops.KV.seq_first(t.transpose(1, 2).contiguous()) for t in (k, v))
    else:
        perm = torch.randperm(B * Hkv * cap, generator=g, device=gpu)
        pools = []
        for t in (k, v):
            pool = torch.empty((B * Hkv * cap, 64, 128), dtype=torch.bfloat16, device=gpu)
            pool[perm] = t.view(-1, 64, 128)
            pools.append(pool)
        pages = perm.to(torch.int32).view(B * Hkv, cap)
        K, V = ops.KV.paged(pools[0], pages), ops.KV.paged(pools[1], pages)
    scale = 1.0 / math.sqrt(128)
    out, lse = ops.attn_decode(q, K, V, lens, scale, cap, Hkv, with_lse=True)
    for b, n in enumerate(lens):
        qf = q[b, 0].float().view(Hkv, Hq // Hkv, 128)
        for h in range(Hkv):
            s = (qf[h] @ k[b, h, :n].float().T.contiguous()) * scale
            ref = torch.softmax(s, -1) @ v[b, h, :n].float()
            err = (out[b, 0].float().view(Hkv, -1, 128)[h] - ref).abs()
            # the attention tolerances: weights are rounded to bf16, an output is a mean under them
            assert err.max() <= 2e-2 and err.mean() <= 2e-3, (b, h, err.max(), err.mean())
            lerr = (lse[b].float().view(Hkv, -1)[h] - torch.logsumexp(s, -1)).abs().max()
            assert lerr <= 4e-3, (b, h, lerr)


@pytest.mark.parametrize("heads_share", [True, False])
def test_decode_of_shared_pages(gpu, heads_share):
    """Requests that share a prefix, among them one that ends inside it and one that shares nothing, in a
    launch that streams what is not shared: bit for bit the output over a copy for each request."""
    lens, prefix, B, Hq, Hkv = [60001, 50003, 1000, 30011], 320, 4, 16, 8
    print(f"case: decode of shared pages lens={lens} heads_share={heads_share}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(11)
    cap = -(-max(lens) // 64)
    q = torch.randn((B, 1, Hq, 128), generator=g, device=gpu).to(torch.bfloat16)
    pages = torch.arange(B * Hkv * cap, dtype=torch.int32, device=gpu).view(B, Hkv, cap)
    for h in range(Hkv):
        if heads_share or h % 2:
            pages[1, h, :prefix] = pages[0, h, :prefix]
            pages[2, h, :prefix] = pages[0, h, :prefix]
    pages[2, :, -(-lens[2] // 64):] = -1  # unmapped
    pages[3, :, -(-lens[3] // 64):] = pages[0, :, -(-lens[3] // 64):]  # left over past the end
    pools = [torch.randn((B * Hkv * cap, 64, 128), generator=g, device=gpu).to(torch.bfloat16) for _ in range(2)]
    own = [t[pages.clamp(min=0).long().view(-1)].view(B, Hkv, cap * 64, 128) for t in pools]
    args = (lens, 1.0 / math.sqrt(128), cap, Hkv)
    out, lse = ops.attn_decode(q, *(ops.KV.paged(t, pages.view(B * Hkv, cap)) for t in pools), *args, with_lse=True)
    want, want_lse = ops.attn_decode(q, *(ops.KV.heads_first(t) for t in own), *args, with_lse=True)
    assert sum(lens) * Hkv * 512 >= 320 << 20
    assert torch.equal(out, want) and torch.equal(lse, want_lse)
    for b, n in enumerate(lens):
        for h in range(0, Hkv, 3):
            s = (q[b, 0, 2 * h:2 * h + 2].float() @ own[0][b, h, :n].float().T.contiguous()) * args[1]
            err = (out[b, 0, 2 * h:2 * h + 2].float() - torch.softmax(s, -1) @ own[1][b, h, :n].float()).abs()
            assert err.max() <= 2e-2 and err.mean() <= 2e-3, (b, h, err.max(), err.mean())


def test_decode_of_an_expanded_cache(gpu):
    """One cache read by every request (stride 0) gives each of them that cache's result."""
    print("case: decode of an expanded cache", flush=True)
    B, n, Hq, Hkv = 8, 24011, 16, 4
    g = torch.Generator(device=gpu).manual_seed(12)
    q = torch.randn((B, 1, Hq, 128), generator=g, device=gpu).to(torch.bfloat16)
    k, v = (torch.randn((1, Hkv, -(-n // 64) * 64, 128), generator=g, device=gpu).to(torch.bfloat16) for _ in range(2))
    args = (1.0 / math.sqrt(128), -(-n // 64), Hkv)
    many = ops.attn_decode(q, *(ops.KV.heads_first(t.expand(B, -1, -1, -1)) for t in (k, v)), [n] * B, *args)
    copies = ops.attn_decode(q, *(ops.KV.heads_first(t.repeat(B, 1, 1, 1)) for t in (k, v)), [n] * B, *args)
    assert B * n * Hkv * 512 >= 320 << 20 and torch.equal(many, copies)
