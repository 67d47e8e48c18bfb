"""Entry points that do in one launch what several did: q and k rotated together, decode tokens
appended through the page table, page tables written beside 128-token block tables."""
from __future__ import annotations

import pytest
import torch

from compactattention_amd import ops
from compactattention_amd.kv_cache import PagedKVCache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,Hq,Hkv", [(1, 32, 8), (3, 17, 16), (130, 4, 1)])
def test_rope_qk_equals_two_calls(gpu, L, Hq, Hkv):
    print(f"case: rope_qk L={L} Hq={Hq} Hkv={Hkv}", flush=True)
    g = torch.Generator().manual_seed(L + Hq)
    x = torch.randn((2, L, (Hq + Hkv) * 128), generator=g).to(torch.bfloat16).to(gpu)
    q, k = x.split([Hq * 128, Hkv * 128], -1)
    q, k = q.view(2, L, Hq, 128), k.view(2, L, Hkv, 128)
    cos, sin = (torch.randn((L, 128), generator=g).to(gpu) for _ in range(2))
    qo, ko = ops.rope_qk(q, k, cos, sin)
    assert torch.equal(qo, ops.rope(q, cos, sin)) and torch.equal(ko, ops.rope(k, cos, sin))


@pytest.mark.parametrize("strided", ["dense", "heads_of_a_wider_row", "odd_strides", "misaligned"])
def test_append_tokens_matches_indexing(gpu, strided):
    """Tokens on both sides of block edges, one and many at a time, next to a CPU cache's indexing;
    rows the kernel cannot read in place (odd strides, a start that is not 16-byte aligned) go through a copy."""
    print(f"case: append_tokens {strided}", flush=True)
    g = torch.Generator().manual_seed(5)
    dev, host = PagedKVCache(2, 3, 64, gpu), PagedKVCache(2, 3, 64, "cpu")
    for n in (1, 62, 1, 1, 130, 5, 64):
        x = torch.randn((2, n, 3, 2 * 128 + (1 if strided == "odd_strides" else 0)), generator=g).to(torch.bfloat16)
        k, v = x[..., :128], x[..., 128:256]
        if strided == "dense":
            k, v = k.contiguous(), v.contiguous()
        xg = x.to(gpu)
        kg, vg = (k.to(gpu), v.to(gpu)) if strided == "dense" else (xg[..., :128], xg[..., 128:256])
        if strided == "misaligned":  # contiguous tensors that start 2 bytes into an allocation
            kg, vg = (torch.cat((t.new_zeros(1), t.reshape(-1)))[1:].view(t.shape) for t in (kg, vg))
            assert kg.is_contiguous() and kg.data_ptr() % 16 != 0
        assert dev.append_tokens(kg, vg) == host.append_tokens(k, v)
    assert torch.equal(dev.k_hf().cpu(), host.k_hf()) and torch.equal(dev.v_hf().cpu(), host.v_hf())


@pytest.mark.parametrize("kb64", [44, 45])
@pytest.mark.parametrize("slack", [0, 3])
def test_page_tables_beside_block_tables(gpu, kb64, slack):
    print(f"case: union pages kb64={kb64} slack={slack}", flush=True)
    B, Hkv, G, Qb = 2, 3, 4, 3
    cap = -(-kb64 // 2)
    P = [cap - Qb] * B
    g = torch.Generator().manual_seed(kb64)
    rowmask = torch.randint(0, 1 << 31, (B, Hkv * G, Qb, ops.words_for(cap)), generator=g, dtype=torch.int32)
    for _ in range(3):  # sparse masks
        rowmask &= torch.randint(0, 1 << 31, rowmask.shape, generator=g, dtype=torch.int32)
    table, counts, _, _, pages, pcounts = ops.union_compact(rowmask.to(gpu), P, Hkv, cap, last_n_block=1,
                                                            pages=(kb64, kb64 + slack))
    t1, c1, _, _ = ops.union_compact(rowmask.to(gpu), P, Hkv, cap, last_n_block=1)
    assert torch.equal(table, t1) and torch.equal(counts, c1)
    table, counts = table.cpu(), counts.cpu()
    for r in range(B * Hkv):
        want = [p for b in table[r, :counts[r]].tolist() for p in (2 * b, 2 * b + 1) if p < kb64]
        assert pages[r].tolist() == want + [-1] * (kb64 + slack - len(want))
        assert int(pcounts[r]) == len(want)
    with pytest.raises(Exception, match="key_pages"):
        ops.union_compact(rowmask.to(gpu), P, Hkv, cap, pages=(kb64 + 2, kb64 + 2))


@pytest.mark.parametrize("n", [2048, 8192, 8200])
@pytest.mark.parametrize("residual", [False, True])
def test_rmsnorm_same_rows_in_launches_of_any_size(gpu, n, residual):
    """Launches above the size that is streamed past the caches give the rows of launches below it."""
    print(f"case: rmsnorm n={n} residual={residual}", flush=True)
    rows = (8 << 20) // n + 1
    g = torch.Generator(device=gpu).manual_seed(n)
    x, r = (torch.randn((rows, n), generator=g, device=gpu).to(torch.bfloat16) for _ in range(2))
    w = torch.randn((n,), generator=g, device=gpu).to(torch.bfloat16)
    norm = lambda a, b: torch.stack(ops.rmsnorm(a, w, 1e-5, residual=b)) if residual else ops.rmsnorm(a, w, 1e-5)  # noqa: E731
    whole = norm(x, r)
    for part in (slice(0, rows - 1), slice(rows - 1, rows), slice(3, 70)):
        assert torch.equal(whole[..., part, :], norm(x[part], r[part]))


@pytest.mark.parametrize("n", [1024, 2040, 2048, 4096])
@pytest.mark.parametrize("elements", [2 << 20, 6 << 20])
def test_rmsnorm_around_its_streamed_sizes(gpu, n, elements):
    """Launches of one row less than a size from which rows are streamed, of that size and one row more."""
    print(f"case: rmsnorm n={n} elements={elements}", flush=True)
    rows = -(-elements // n)
    g = torch.Generator(device=gpu).manual_seed(n)
    x, r = (torch.randn((rows + 1, n), generator=g, device=gpu).to(torch.bfloat16) for _ in range(2))
    w = torch.randn((n,), generator=g, device=gpu).to(torch.bfloat16)
    few = torch.cat([torch.stack(ops.rmsnorm(x[i:i + 400], w, 1e-5, residual=r[i:i + 400]))
                     for i in range(0, rows + 1, 400)], 1)
    for m in (rows - 1, rows, rows + 1):
        assert torch.equal(torch.stack(ops.rmsnorm(x[:m], w, 1e-5, residual=r[:m])), few[:, :m])
