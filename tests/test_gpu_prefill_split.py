"""Prefill launches of at most half as many query blocks as the device has
compute units split their keys over work-groups and merge the pieces: against
the fp32 oracle, over the key sources, at the edges of pieces, bands and windows."""
from importlib import import_module

import pytest
import torch

from helpers import assert_lse_close, assert_out_close
from oracle import attn_ref

pytestmark = pytest.mark.gpu


def _runs(lens, prior, hq, hkv, seed, source, wl, E=0, window=0):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(s, generator=g).to(torch.bfloat16)  # noqa: E731
    T = sum(lens)
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    a = dict(q=r(T, hq, 128), k=None, v=None, cu_seqlens=cu, scale=128 ** -0.5,
             window=window)
    if source != "paged":
        a.update(k=r(T, hkv, 128), v=r(T, hkv, 128))
    if source != "packed":
        table, P = wl.paged_layout(lens, g, prior=prior)
        a.update(prior_lens=torch.tensor(prior, dtype=torch.int32),
                 k_pool=r(P, 16, hkv, 128), v_pool=r(P, 16, hkv, 128),
                 block_table=table)
    if source == "ring":
        a["table_wrap"] = a["block_table"].shape[1]
    if E:
        a["rel"] = torch.randn((T, hq, E), generator=g).to(torch.bfloat16)
    return a


def _check(tm, dev, a, what, split=True):
    lens = (a["cu_seqlens"][1:] - a["cu_seqlens"][:-1])
    ref_o, ref_l = attn_ref.prefill_varlen(**a)
    d = {k: v.to(dev) if torch.is_tensor(v) else v for k, v in a.items()}
    bt = a.get("block_table")
    n = tm._lib.load().tmopt_attn_prefill_workspace_size(
        lens.numel(), int(lens.max()), a["q"].shape[1],
        (a["k_pool"] if a["k"] is None else a["k"]).shape[-2],
        0 if bt is None else bt.shape[1], a.get("table_wrap", 0), a["window"])
    assert (n > 0) == split, (what, n)
    out, lse = tm.prefill_varlen(**d)
    torch.cuda.synchronize()
    assert_out_close(out, ref_o, what)
    assert_lse_close(lse, ref_l, what)
    return d, out, lse


@pytest.mark.parametrize("source", ["paged", "mixed"])
@pytest.mark.parametrize("lens,prior", [
    ([1], [2000]), ([31], [993]), ([32], [1248]), ([33], [1311]),
    ([200], [3000]), ([5, 40], [1500, 0]), ([64, 1, 17], [10, 4000, 700])])
def test_short_chunks_after_long_context(tm, dev, source, lens, prior):
    """From one query to 200, after contexts of up to 4000 keys: items of one
    piece, written in place, beside items of many."""
    wl = import_module("tm-opt_amd.workloads")
    for i, (hq, hkv) in enumerate([(32, 4), (8, 8), (16, 2), (3, 1)]):
        _check(tm, dev, _runs(lens, prior, hq, hkv, 50 + i, source, wl),
               f"{source} {lens} after {prior}, {hq}/{hkv}")


@pytest.mark.parametrize("lens", [[3072], [3100], [2017, 3050]])
@pytest.mark.parametrize("window", [0, 3000])
def test_few_short_prompts(tm, dev, lens, window):
    wl = import_module("tm-opt_amd.workloads")
    a = _runs(lens, [0] * len(lens), 2, 1, 60, "packed", wl, window=window)
    _check(tm, dev, a, f"prompts {lens} w={window}")


@pytest.mark.parametrize("E", [1, 70, 512, 1024, 5000])
@pytest.mark.parametrize("hq,hkv", [(16, 2), (8, 2)])
def test_bias_band_across_pieces(tm, dev, E, hq, hkv):
    """Pieces past the bias band run without a bias, the others with one; the
    band's end falls inside a piece, at its edge, or past every key."""
    wl = import_module("tm-opt_amd.workloads")
    a = _runs([70, 33], [1981, 900], hq, hkv, 61, "mixed", wl, E=E)
    _check(tm, dev, a, f"bias E={E} {hq}/{hkv}")


@pytest.mark.parametrize("W,prior", [(1280, 200), (1280, 1280), (1280, 5000),
                                     (2048, 2500)])
def test_ring_chunk(tm, dev, W, prior):
    wl = import_module("tm-opt_amd.workloads")
    g = torch.Generator().manual_seed(62)
    T, hq, hkv, per = 96, 16, 2, W // 16
    a = _runs([T], [0], hq, hkv, 62, "mixed", wl, E=W, window=W)
    a.update(prior_lens=torch.tensor([prior], dtype=torch.int32),
             block_table=torch.randperm(per, generator=g).int()[None],
             k_pool=torch.randn((per, 16, hkv, 128), generator=g).bfloat16(),
             v_pool=torch.randn((per, 16, hkv, 128), generator=g).bfloat16(),
             table_wrap=per)
    _check(tm, dev, a, f"ring W={W} prior={prior}")


def test_split_repeats_bitwise_and_matches_one_launch(tm, dev):
    """The merge order is fixed; the unsplit entry point (no workspace) gives
    the same result to the rounding of one bf16 store. A launch of more
    items than half the compute units does not split; a short workspace is refused;
    a rejected launch is NaN whole."""
    wl = import_module("tm-opt_amd.workloads")
    a = _runs([130], [2500], 32, 4, 63, "paged", wl)
    d, out, lse = _check(tm, dev, a, "repeat")
    again = tm.prefill_varlen(**d)
    assert torch.equal(again[0], out) and torch.equal(again[1], lse)
    attn = import_module("tm-opt_amd.attn")
    size = attn._prefill_workspace_size
    attn._prefill_workspace_size = lambda *a: 0
    try:
        one = tm.prefill_varlen(**d)
    finally:
        attn._prefill_workspace_size = size
    torch.cuda.synchronize()
    # two correct roundings of O to bf16 differ by one ulp at most (2^-7 of
    # the value); the rounding of P adds 2^-9 of the values' sums
    assert ((one[0].float() - out.float()).abs() <=
            2 ** -7 * out.float().abs() + 2e-3).all()
    assert (one[1] - lse).abs().max() <= 1e-4
    rej = torch.ones(1, dtype=torch.int32, device=dev)
    o, l = tm.prefill_varlen(**d, reject=rej)
    assert torch.isnan(o).all() and torch.isnan(l).all()
    size = tm._lib.load().tmopt_attn_prefill_workspace_size
    assert size(1, 3000, 32, 4, 0, 0, 0) == 0
    assert size(1, 130, 32, 4, 79, 0, 0) > 0    # 1264 + 130 keys
    assert size(1, 16, 32, 4, 58, 0, 0) == 0    # 944 keys
    with pytest.raises(tm.TmoptError) as e:
        real = tm._lib.call
        try:
            tm._lib.call = lambda name, *x: real(
                name, *(x[:-2] + (1024,) + x[-1:])
                if name.endswith("_split") else x)
            tm.prefill_varlen(**d)
        finally:
            tm._lib.call = real
    assert e.value.status == tm._lib.TMOPT_EWORKSPACE


@pytest.mark.parametrize("lens,prior", [
    ([64, 256], [7936, 7680]), ([96, 256], [7808, 6720]), ([7], [40])])
def test_merge_reads_what_was_written(tm, dev, lens, prior):
    """Lengths at which the fp32 rule for the number of pieces sits on a
    rounding edge (12 or 13 of them with and without an fma; found with both
    forms on the CPU), and a launch whose items all stay whole, over a scratch
    full of NaN: the merge takes exactly the pieces that were left for it."""
    wl = import_module("tm-opt_amd.workloads")
    a = _runs(lens, prior, 16, 2, 64, "paged", wl)
    if lens == [7]:
        a["block_table"] = torch.nn.functional.pad(a["block_table"], (0, 100))
    real, held = tm._lib.call, []

    def call(name, *x):
        if name.endswith("_split"):
            held.append(torch.full((x[-2] // 4 + 4,), float("nan"),
                                   device=dev))
            x = x[:-3] + (held[0].data_ptr(),) + x[-2:]
        return real(name, *x)
    tm._lib.call = call
    try:
        _check(tm, dev, a, f"{lens} after {prior}")
    finally:
        tm._lib.call = real
    assert held


@pytest.mark.parametrize("prior", [1500, 4000])
def test_infinite_values(tm, dev, prior):
    """An infinity in V that every query sees, in the last piece, is one in
    each of their outputs of that dim and KV head, and no NaN anywhere."""
    wl = import_module("tm-opt_amd.workloads")
    a = _runs([40], [prior], 16, 2, 71, "paged", wl)
    a["v_pool"][int(a["block_table"][0, prior // 16]), 0, 1, 3] = float("inf")
    a["scale"] = 0.01            # no probability of that key rounds to zero
    d = {k: v.to(dev) if torch.is_tensor(v) else v for k, v in a.items()}
    out, _ = tm.prefill_varlen(**d)
    torch.cuda.synchronize()
    want = torch.zeros(out.shape, dtype=torch.bool)
    want[:, 8:, 3] = True
    out = out.cpu()
    assert torch.equal(out.isinf(), want) and not out.isnan().any()
