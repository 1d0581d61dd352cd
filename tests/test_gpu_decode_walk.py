"""The decode walk's edges against the fp32 oracle: ranges of more page ids
than the kernel keeps in LDS, rows of a window's first page that lie before
the window, bias rows at every alignment, and the shapes of the merge."""
from importlib import import_module

import pytest
import torch

from helpers import assert_lse_close, assert_out_close
from oracle import attn_ref

pytestmark = pytest.mark.gpu


def _check(tm, dev, case, what, rel=None, **kw):
    ref_o, ref_l = attn_ref.decode_paged(
        case.q, case.k_pool, case.v_pool, case.block_table, case.ctx_lens,
        case.scale, window=case.window, rel=rel)
    c = case.to(dev)
    out, lse = tm.decode_paged(
        c.q, c.k_pool, c.v_pool, c.block_table, c.ctx_lens, c.scale,
        window=c.window, rel=None if rel is None else rel.to(dev), **kw)
    torch.cuda.synchronize()
    assert_out_close(out, ref_o, what)
    assert_lse_close(lse, ref_l, what)


@pytest.mark.parametrize("ctx", [[63990, 40], [64017, 1, 0, 33],
                                 [70, 66000, 65]])
def test_range_beyond_the_kept_page_ids(tm, dev, ctx):
    """One work-group walks everything: 4000 page ids are kept without a bias
    (64,000 tokens), 1500 with one (24,000), the rest are looked up on the
    way. The last kept page is a step's first or second one, or a sequence's
    last."""
    wl = import_module("tm-opt_amd.workloads")
    g = torch.Generator().manual_seed(41)
    case = wl.make_decode("ids", 41, len(ctx), 0, 0, hq=4, hkv=1, ctx=ctx)
    _check(tm, dev, case, f"ids {ctx}", num_workgroups=1)
    ctx = [max(0, c - 40000) if c > 40000 else c for c in ctx]
    case = wl.make_decode("ids", 42, len(ctx), 0, 0, hq=4, hkv=1, ctx=ctx)
    rel = (torch.randn((len(ctx), 4, 300), generator=g) * 0.5).bfloat16()
    _check(tm, dev, case, f"ids + bias {ctx}", rel, num_workgroups=1)


@pytest.mark.parametrize("window", [1, 15, 17, 31, 100])
def test_window_starts_inside_a_page(tm, dev, window):
    """Rows of the window's first page that lie before the window hold NaN:
    they are outside the loads' resource, in K and in V."""
    wl = import_module("tm-opt_amd.workloads")
    ctx = [window + k for k in range(0, 34, 3)] + [1, 16, 333]
    case = wl.make_decode("win", 43, len(ctx), 0, 0, window, ctx=ctx)
    for b, n in enumerate(ctx):
        first = max(0, n - window)
        for p in range(first // 16 * 16, first):
            page = int(case.block_table[b, p // 16])
            case.k_pool[page, p % 16] = float("nan")
            case.v_pool[page, p % 16] = float("nan")
    _check(tm, dev, case, f"window {window}", min_pages=1)


@pytest.mark.parametrize("hq,hkv", [(4, 4), (6, 1), (8, 1), (16, 1), (12, 1),
                                    (40, 2)])
@pytest.mark.parametrize("E", [1, 2, 7, 33, 64, 65])
def test_bias_rows_at_every_alignment(tm, dev, hq, hkv, E):
    """E odd puts every other row mid-dword; head 0 of sequence 0 starts at
    the first byte of the tensor, the last head ends at its last one;
    contexts around E have steps inside, across and past the band."""
    wl = import_module("tm-opt_amd.workloads")
    g = torch.Generator().manual_seed(E)
    ctx = [1, 2, 3, 4, 5, 16, 31, 32, 33, 48, 63, 64, 65, 66, 95, 130]
    case = wl.make_decode("rel", 44, len(ctx), 0, 0, hq=hq, hkv=hkv, ctx=ctx)
    rel = torch.randn((len(ctx), hq, E), generator=g).bfloat16()
    _check(tm, dev, case, f"E={E} {hq}/{hkv}", rel, min_pages=2)


@pytest.mark.parametrize("B,hq,hkv,pages", [
    (1, 32, 4, 190), (1, 32, 4, 500), (1, 7, 1, 33), (2, 9, 3, 400), (5, 16, 2, 90),
    (23, 32, 4, 40), (24, 32, 4, 40), (64, 8, 8, 12)])
def test_merge_shapes(tm, dev, B, hq, hkv, pages):
    """Shares of one page and more (min_pages 1) over grids of 7 to 200
    work-groups: from a merge of 190 pieces, one per page, by 32 groups per
    head to one of two pieces, an odd number of heads per work-group, more
    groups than pieces, sequences that need no merge beside ones that do."""
    wl = import_module("tm-opt_amd.workloads")
    g = torch.Generator().manual_seed(B)
    ctx = torch.randint(1, 16 * pages, (B,), generator=g)
    ctx[0] = 16 * pages
    if B > 2:
        ctx[1] = 3
    case = wl.make_decode("merge", 45, B, 0, 0, hq=hq, hkv=hkv, ctx=ctx)
    for wgs in (0, 7, 64, 200):
        _check(tm, dev, case, f"merge B={B} wgs={wgs}", min_pages=1,
               num_workgroups=wgs)


@pytest.mark.parametrize("HQ,HK,E", [(64, 8, 1024), (12, 4, 33), (4, 4, 64)])
def test_flat_rows_in_place(tm, dev, HQ, HK, E):
    """decode_flat against decode_paged over the table made of the same rows:
    bitwise (same kernel, same split); Lg a multiple of 16 and not, positions
    past Lg (their pages are absent), row ids outside the pool."""
    g = torch.Generator().manual_seed(46)
    pos = torch.tensor([0, 15, 16, 700, 40, 1535, 1600, 333])
    B, P = pos.shape[0], 900
    kp = torch.randn((P, 16, HK, 128), generator=g).bfloat16().to(dev)
    vp = torch.randn((P, 16, HK, 128), generator=g).bfloat16().to(dev)
    q = torch.randn((B, HQ, 128), generator=g).bfloat16().to(dev)
    rel = torch.randn((B, HQ, E), generator=g).bfloat16().to(dev)
    for Lg in (1536, 1500, 17):
        npg = -(-Lg // 16)
        table = torch.randperm(P, generator=g)[:B * npg].view(B, npg)
        table[3, npg // 2] = P + 5
        j = torch.arange(Lg)
        flat = table[:, j // 16] * 16 + (j % 16)[None]
        flat = flat.masked_fill(j[None] > pos[:, None], 0).contiguous().to(dev)
        t, n = tm.decode_table_from_flat(flat, pos.to(dev))
        for r in (rel, None):
            want = tm.decode_paged(q, kp, vp, t, n, 1 / 128, rel=r)
            got = tm.decode_flat(q, kp, vp, flat, pos.to(dev), 1 / 128,
                                 rel=r, return_lse=True)
            torch.cuda.synchronize()
            assert torch.equal(got[0], want[0]), (Lg, r is None)
            assert torch.equal(got[1], want[1]), (Lg, r is None)


def test_flat_rows_beyond_the_kept_page_ids(tm, dev):
    """One work-group over more than 1500 pages of flat rows: the later ids
    are looked up on the way."""
    g = torch.Generator().manual_seed(47)
    pos = torch.tensor([25000, 600])
    Lg, P = 25001, 3200
    kp = torch.randn((P, 16, 1, 128), generator=g).bfloat16().to(dev)
    vp = torch.randn((P, 16, 1, 128), generator=g).bfloat16().to(dev)
    q = torch.randn((2, 4, 128), generator=g).bfloat16().to(dev)
    rel = torch.randn((2, 4, 100), generator=g).bfloat16().to(dev)
    table = torch.randperm(P, generator=g)[:2 * 1563].view(2, 1563)
    j = torch.arange(Lg)
    flat = (table[:, j // 16] * 16 + (j % 16)[None]).contiguous().to(dev)
    t, n = tm.decode_table_from_flat(flat, pos.to(dev))
    want = tm.decode_paged(q, kp, vp, t, n, 1 / 128, rel=rel,
                           num_workgroups=1)
    got = tm.decode_flat(q, kp, vp, flat, pos.to(dev), 1 / 128, rel=rel,
                         num_workgroups=1, return_lse=True)
    torch.cuda.synchronize()
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("B,pages", [(1, 500), (5, 90), (24, 40)])
def test_merge_of_infinite_values(tm, dev, B, pages):
    """An infinity in V is one in that dim's output of the heads that read
    it, whatever the number of pieces the merge rounds up to, and no NaN."""
    wl = import_module("tm-opt_amd.workloads")
    case = wl.make_decode("inf", 48, B, 0, 0, hq=8, hkv=2,
                          ctx=[16 * pages] * B)
    for b in range(B):
        case.v_pool[int(case.block_table[b, 0]), 5, 1, 3] = float("inf")
    c = case.to(dev)
    want = torch.zeros((B, 8, 128), dtype=torch.bool)
    want[:, 4:, 3] = True
    for wgs in (0, 7, 64):
        out, _ = tm.decode_paged(c.q, c.k_pool, c.v_pool, c.block_table,
                                 c.ctx_lens, 0.01, min_pages=1,
                                 num_workgroups=wgs)
        torch.cuda.synchronize()
        out = out.cpu()
        assert torch.equal(out.isinf(), want), wgs
        assert not out.isnan().any(), wgs


def test_merge_of_more_heads_than_a_grid_dimension(tm, dev):
    """65,538 query heads over 64 ranges: the merge's grid holds heads in its
    y dimension (65,536 at most), eight to a work-group. Against the launch
    that splits nothing, to two roundings of O to bf16 (2^-7 of the value) and
    of P (2^-9 of the values' sums)."""
    g = torch.Generator(device=dev).manual_seed(49)
    HQ, HKV, n = 65538, 32769, 70
    r = lambda *s: torch.randn(s, generator=g, device=dev,  # noqa: E731
                               dtype=torch.bfloat16)
    q, kp, vp = r(1, HQ, 128), r(5, 16, HKV, 128), r(5, 16, HKV, 128)
    table = torch.tensor([[3, 0, 4, 2, 1]], dtype=torch.int32, device=dev)
    ctx = torch.tensor([n], dtype=torch.int32, device=dev)
    one = tm.decode_paged(q, kp, vp, table, ctx, 128 ** -0.5,
                          num_workgroups=1)
    out = tm.decode_paged(q, kp, vp, table, ctx, 128 ** -0.5, min_pages=1,
                          num_workgroups=64)
    torch.cuda.synchronize()
    assert ((one[0].float() - out[0].float()).abs() <=
            2 ** -7 * one[0].float().abs() + 1e-2).all()
    assert (one[1] - out[1]).abs().max() <= 1e-4
