"""The launches that prepare a call: K and V whose channel-major rows no
kernel reads in place (tmopt_pack_rows) and a chunk batch's index tensors
(tmopt_chunk_tables), both exact against the torch expressions they stand
for, and the decode ring's grid on both sides of its line."""
import importlib

import pytest
import torch

from helpers import assert_out_close
from oracle import attn_ref

pytestmark = pytest.mark.gpu


def _mod(name):
    return importlib.import_module("tm-opt_amd." + name)


@pytest.mark.parametrize("B,HK,T,pad", [
    (1, 1, 1, 0), (1, 8, 777, 0), (2, 3, 63, 0), (3, 2, 65, 7), (2, 4, 64, 3),
    (1, 16, 130, 1)])
def test_pack_rows_is_the_transpose(tm, dev, B, HK, T, pad):
    """Token counts around the 64-token tile, dim rows at any 2-byte
    alignment (pad), K and V of different strides."""
    g = torch.Generator().manual_seed(7 * B + T)

    def cm(p):
        x = torch.randn((B, HK, 128, T + p), generator=g)
        return x.to(torch.bfloat16).to(dev)[..., p // 2:p // 2 + T]

    k, v = cm(pad), cm(pad + 2)
    kt, vt = k.permute(0, 3, 1, 2), v.permute(0, 3, 1, 2)
    ko, vo = _mod("attn")._pack_rows(kt, vt)
    assert ko.is_contiguous() and vo.is_contiguous()
    assert torch.equal(ko, kt) and torch.equal(vo, vt)
    compat = _mod("compat")
    kr, vr = compat._kv_pair(k.transpose(2, 3), v.transpose(2, 3))
    assert torch.equal(kr, kt) and torch.equal(vr, vt)
    for x, src in ((kr, kt), (vr, vt)):
        assert x.shape == (B, T, HK, 128)
        assert x.data_ptr() == src.data_ptr() or x.is_contiguous()


def test_kv_pair_leaves_what_is_read_in_place(tm, dev):
    """One tensor in place and one not, and token-major rows: as each would
    be alone."""
    compat = _mod("compat")
    odd = torch.randn((1, 2, 128, 77), device=dev).to(torch.bfloat16)
    even = torch.randn((1, 2, 128, 80), device=dev).to(torch.bfloat16)
    odd, even = odd.transpose(2, 3), even.transpose(2, 3)[:, :, :77]
    kr, vr = compat._kv_pair(even, odd)
    assert kr.data_ptr() == even.data_ptr() and vr.is_contiguous()
    assert torch.equal(kr, even.transpose(1, 2))
    assert torch.equal(vr, odd.transpose(1, 2))


@pytest.mark.parametrize("B,S,width", [(1, 1, 1), (3, 3, 255), (2, 1, 256),
                                       (5, 5, 700)])
def test_chunk_tables_are_the_index_expressions(tm, dev, B, S, width):
    """Widths around the 256-entry block, negative slots, more slots than
    runs, rows at a stride wider than the row."""
    attn = _mod("attn")
    g = torch.Generator().manual_seed(B + width)
    rows = 9
    td = torch.randint(-1, 1 << 20, (rows, width + 3), generator=g)
    td = td.to(dev)[:, :width]
    slots = torch.randint(-rows, rows, (B,), generator=g).to(dev)
    prior = torch.randint(0, 5000, (2 * S,), generator=g).to(dev)[::2]
    table, start, cu = attn._chunk_tables(slots, prior, width, td, 41)
    assert torch.equal(table, td[slots].to(torch.int32))
    assert torch.equal(start, prior.to(torch.int32))
    assert cu.tolist() == [0, 41]
    table, start, _ = attn._chunk_tables(slots, prior, width)
    want = slots[:, None] * width + torch.arange(width, device=dev)
    assert torch.equal(table, want.to(torch.int32))
    assert torch.equal(start, prior.to(torch.int32))
    out = torch.full((B,), rows, device=dev)
    table, _, _ = attn._chunk_tables(out, prior, width, td)
    assert (table == -1).all()


@pytest.mark.parametrize("bad", [3, -4, 1 << 40])
@pytest.mark.parametrize("prior", [20, 1500])
def test_slot_outside_the_table_is_rejected(tm, dev, bad, prior):
    """A slot that names no row of the page table (torch's indexing refuses
    it) makes the whole call NaN, in one launch and with split keys, and
    appends nothing for it; slots that count from the end are accepted."""
    rows, width, T = 3, 100, 8
    g = torch.Generator().manual_seed(9)
    r = lambda *s: torch.randn(s, generator=g).bfloat16().to(dev)  # noqa: E731
    q, k, v = r(2 * T, 16, 128), r(2 * T, 2, 128), r(2 * T, 2, 128)
    kp, vp = r(rows * width, 16, 2, 128), r(rows * width, 16, 2, 128)
    td = torch.randperm(rows * width, generator=g).view(rows, width).to(dev)
    cu = torch.tensor([0, T, 2 * T], dtype=torch.int32, device=dev)
    pr = torch.tensor([prior, prior], device=dev)
    for slots in ([bad, 1], [1, bad], [-rows, rows - 1]):
        k0, v0 = kp.clone(), vp.clone()
        out = tm.attn_prefill_chunk_global(
            q, k, v, None, k0, v0, td, torch.tensor(slots, device=dev), pr,
            cu_seqlens=cu, max_seqlen=T)
        torch.cuda.synchronize()
        if bad not in slots:
            assert not out.isnan().any()
            continue
        assert out.isnan().all()
        pages = td[1, prior // 16:(prior + T - 1) // 16 + 1]
        same = torch.ones(rows * width, dtype=torch.bool)
        same[pages.cpu()] = False
        assert torch.equal(k0.cpu()[same], kp.cpu()[same])
        assert torch.equal(v0.cpu()[same], vp.cpu()[same])


@pytest.mark.parametrize("slots", [0, 2])
def test_batch_of_no_chunks(tm, dev, slots):
    """No run (cu_seqlens of one entry), with slots or without: an empty
    output and untouched pools, as before the index tensors were one
    launch."""
    bf = torch.bfloat16
    q = torch.zeros((0, 16, 128), dtype=bf, device=dev)
    k = torch.zeros((0, 2, 128), dtype=bf, device=dev)
    kp, vp = (torch.ones((8, 16, 2, 128), dtype=bf, device=dev)
              for _ in range(2))
    none = torch.zeros(0, dtype=torch.int64, device=dev)
    sl = torch.arange(slots, device=dev)
    kw = dict(cu_seqlens=torch.zeros(1, dtype=torch.int32, device=dev),
              max_seqlen=0)
    out = tm.attn_prefill_chunk_global(
        q, k, k, None, kp, vp, torch.zeros((2, 4), dtype=torch.int64,
                                           device=dev), sl, none, **kw)
    assert out.shape == q.shape
    ring = torch.ones((3, 32, 2, 128), dtype=bf, device=dev)
    out = tm.attn_prefill_chunk_swa(q, k, k, None, ring, ring, sl, none, **kw)
    torch.cuda.synchronize()
    assert out.shape == q.shape
    assert (kp == 1).all() and (vp == 1).all() and (ring == 1).all()


@pytest.mark.parametrize("B,HQ,HK,W", [(1, 64, 16, 512), (38, 64, 16, 128),
                                       (39, 64, 16, 128), (73, 32, 4, 64)])
def test_ring_grid_line(tm, dev, B, HQ, HK, W):
    """attn_swa where whole rings reach few compute units (its rows split
    over the default grid) and where they reach enough, either side of the
    line on 256 units: against the oracle, within 2e-2 + 1e-2 |ref|."""
    g = torch.Generator().manual_seed(B)
    D = 128
    pos = torch.randint(0, 3 * W, (B,), generator=g)
    pool_k, pool_v = ((torch.randn((B + 1, W, HK, D), generator=g) * 0.5).to(
        torch.bfloat16) for _ in range(2))
    slots = torch.randperm(B, generator=g)
    q = torch.randn((B, HQ, D), generator=g).to(torch.bfloat16)
    rel = (torch.randn((B, HQ, W), generator=g) * 0.5).to(torch.bfloat16)
    ref, _ = attn_ref.decode_reference_semantics(q, pool_k, pool_v, slots,
                                                 pos, rel, W)
    out = tm.attn_swa(q.to(dev), pool_k.to(dev), pool_v.to(dev),
                      slots.to(dev), pos.to(dev), rel.to(dev))
    assert_out_close(out, ref, "ring")
