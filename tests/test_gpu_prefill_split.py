"""GPU parity of the KV-split form of the prefill attention (axk_paged_prefill_split: few row blocks over a long history)
at the edges of its pieces: histories at, below and above whole pieces of 256 tokens, row blocks whose rows end in
the middle of a wave, pages outside the pool inside a piece, and scales of either sign.

Bar: bf16 outputs within rel 2e-2 / abs 1e-2 of the fp32 oracle; the split and unsplit forms (the same products, summed
in another order and rounded to bf16 once) within two bf16 roundings, rel 2 * 2^-8, of each other beside the
probabilities' own rounding (abs 1e-2).
"""
import pytest
import torch

from axk import _lib, attention, configs, layer
from oracle import paged_attn as pa

pytestmark = pytest.mark.gpu
TOL = dict(rtol=2e-2, atol=1e-2)


def _dev(c, dev):
    return {k: (v.to(dev) if torch.is_tensor(v) else v) for k, v in c.items()}


def _call(c, dev, split, scale, status=None):
    d = _dev(c, dev)
    t, hq, hd = d["q"].shape
    p, _, page, hkv, _ = d["cache"].shape
    b = len(c["qlens"])
    out = torch.full_like(d["q"], float("nan"))
    args = [d[n].data_ptr() for n in ("q", "cache", "qo_indptr", "indptr", "indices", "last_page_len")]
    tail = (out.data_ptr(), b, t, hq, hkv, hd, page, p, scale, _lib.ptr(status))
    if split:
        n = _lib.load().axk_paged_prefill_workspace_size(b, t, hq, hkv, hd)
        assert n > 0, "the case does not split"
        ws = torch.full((n,), 255, dtype=torch.uint8, device=dev)
        _lib.call("axk_paged_prefill_split", *args, *tail, ws.data_ptr(), n, _lib.stream_of(out))
    else:
        _lib.call("axk_paged_prefill", *args, *tail, _lib.stream_of(out))
    return out.cpu()


@pytest.mark.parametrize("qlens,kv_lens,hq,hkv,d,page", [
    ([1], [256], 16, 2, 256, 64),              # exactly one piece: unsplit inside a splitting call
    ([1], [257], 16, 2, 256, 64),              # a second piece of one token
    ([4, 3], [4096, 511], 32, 4, 256, 64),     # draft rows, one sequence of two pieces
    ([33, 1, 0], [3000, 1, 40], 8, 2, 128, 16),  # pairs crossing pages, a one-token sequence, an empty query range
    ([17], [20000], 16, 1, 64, 256),           # 64 splits of a long history, head dim 64
    ([100], [5001], 12, 3, 128, 32),           # three KV heads: no whole XCDs per head; group 4
    ([300], [700], 16, 2, 256, 48),            # row blocks of several pieces, pages of three tiles
    ([20, 20], [20, 1300], 24, 2, 128, 128),   # group 12: rows straddle tokens
])
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_split_matches_oracle_and_unsplit(dev, qlens, kv_lens, hq, hkv, d, page, sign):
    g = torch.Generator().manual_seed(sum(kv_lens) + hq + d)
    c = configs.prefill_case(qlens, kv_lens, hq, hkv, d, page, g, extra_pages=2)
    print(f"case qlens={qlens} kv_lens={kv_lens} hq={hq} hkv={hkv} d={d} page={page} sign={sign}", flush=True)
    scale = sign * c["scale"]
    got = _call(c, dev, True, scale)
    ref = pa.paged_prefill(c["q"], c["cache"], c["qo_indptr"], c["indptr"], c["indices"], c["last_page_len"], scale)
    torch.testing.assert_close(got.float(), ref.to(torch.bfloat16).float(), **TOL)
    torch.testing.assert_close(got.float(), _call(c, dev, False, scale).float(), rtol=2 ** -7, atol=1e-2)
    assert torch.equal(got.view(torch.int16), _call(c, dev, True, scale).view(torch.int16))  # deterministic


@pytest.mark.parametrize("qlens,kv_lens,hq,hkv,d,page", [
    ([64], [4096], 16, 2, 256, 64),
    ([4, 3, 2], [4096, 511, 900], 32, 4, 256, 64),
    ([33, 1], [3000, 300], 8, 2, 128, 16),  # pairs crossing pages; pieces past the first 64 pages of a table
    ([17], [9000], 16, 1, 64, 16),
])
def test_split_rounds_as_unsplit(dev, qlens, kv_lens, hq, hkv, d, page):
    """A split's probabilities are rounded to bf16 against the sequence's own reference maximum, as the unsplit form's are,
    so the two differ by fp32 sums alone: fewer than 1 % of the outputs round to the neighbouring bf16 value, and the
    difference is below sqrt(0.01) 2^-8 of the output."""
    g = torch.Generator().manual_seed(sum(kv_lens) + d)
    c = configs.prefill_case(qlens, kv_lens, hq, hkv, d, page, g, extra_pages=2)
    print(f"case qlens={qlens} kv_lens={kv_lens} hq={hq} hkv={hkv} d={d} page={page}", flush=True)
    split, whole = (_call(c, dev, form, c["scale"]).double() for form in (True, False))
    assert float((split - whole).norm() / whole.norm()) <= 0.1 * 2 ** -8


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("kv", [30, 32, 33, 70])
def test_output_8_byte_aligned(dev, d, kv):
    """Contexts of one pair of tiles, of a whole pair and of a token more; an output that is 8-byte aligned only (its rows
    then leave in 8-byte pieces) holds the same bits as an aligned one."""
    g = torch.Generator().manual_seed(d + kv)
    c = _dev(configs.prefill_case([5, 2], [kv, kv + 3], 8, 2, d, 16, g), dev)
    args = (c["q"], c["cache"], c["qo_indptr"], c["indptr"], c["indices"], c["last_page_len"])
    want = attention.paged_prefill(*args)
    ref = pa.paged_prefill(*(t.cpu() for t in args), c["scale"])
    torch.testing.assert_close(want.float().cpu(), ref.to(torch.bfloat16).float(), **TOL)
    pool = torch.full((c["q"].numel() + 8,), float("nan"), dtype=torch.bfloat16, device=dev)
    out = pool[4:4 + c["q"].numel()].view_as(c["q"])
    assert out.data_ptr() % 16 == 8
    attention.paged_prefill(*args, output=out)
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
    assert pool[:4].isnan().all() and pool[4 + c["q"].numel():].isnan().all()


def test_split_zero_scale_is_the_mean(dev):
    g = torch.Generator().manual_seed(8)
    c = configs.prefill_case([2], [900], 8, 2, 128, 64, g)
    print("case zero scale", flush=True)
    ref = pa.paged_prefill(c["q"], c["cache"], c["qo_indptr"], c["indptr"], c["indices"], c["last_page_len"], 0.0)
    torch.testing.assert_close(_call(c, dev, True, 0.0).float(), ref.to(torch.bfloat16).float(), **TOL)


@pytest.mark.parametrize("split", [False, True])
def test_bad_pages_hold_no_tokens(dev, split):
    """Pages outside the pool count as absent even where page 0 of the pool holds NaN: the output equals the oracle's on
    the sequence without them."""
    g = torch.Generator().manual_seed(9)
    page = 16
    c = configs.prefill_case([3], [1200], 8, 2, 128, page, g, extra_pages=1)
    spare = [p for p in range(c["cache"].shape[0]) if p not in set(c["indices"].tolist())][0]
    idx = c["indices"].clone()
    idx[idx == 0] = spare  # page 0 leaves the table ...
    c["cache"][spare] = c["cache"][0]
    c["cache"][0] = float("nan")  # ... and holds NaN
    bad = [2, 3, 30, 45]  # a whole pair of tiles, and single tiles of a pair
    keep = [i for i in range(len(idx)) if i not in bad]
    good = c["cache"][idx[keep].long()]
    dense = dict(c, cache=good.contiguous(), indices=torch.arange(len(keep), dtype=torch.int32),
                 indptr=torch.tensor([0, len(keep)], dtype=torch.int32))
    ref = pa.paged_prefill(dense["q"], dense["cache"], dense["qo_indptr"], dense["indptr"], dense["indices"],
                           dense["last_page_len"], c["scale"])
    idx[bad] = torch.tensor([-1, 10 ** 6, c["cache"].shape[0], -7], dtype=torch.int32)
    c["indices"] = idx
    status = torch.zeros(1, dtype=torch.int32, device=dev)
    print(f"case bad pages split={split}", flush=True)
    got = _call(c, dev, split, c["scale"], status)
    torch.testing.assert_close(got.float(), ref.to(torch.bfloat16).float(), **TOL)
    assert int(status.item()) == 1


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("d,pages,last", [(128, 75, 16), (256, 21, 5)])
def test_bad_last_page_of_an_odd_count(dev, d, pages, last, split):
    """The last tile of an odd count is paired with itself: where its page is outside the pool and page 0 of the pool (whose
    bytes it is loaded from) holds NaN, neither of the two reaches the output."""
    g = torch.Generator().manual_seed(12)
    page, t, hq, hkv = 16, 3, 8, 2
    kv = (pages - 1) * page + last
    c = configs.prefill_case([t], [kv], hq, hkv, d, page, g, extra_pages=1)
    spare = [p for p in range(c["cache"].shape[0]) if p not in set(c["indices"].tolist())][0]
    idx = c["indices"].clone()
    idx[idx == 0] = spare
    c["cache"][spare] = c["cache"][0]
    c["cache"][0] = float("nan")
    idx[-1] = c["cache"].shape[0]
    c["indices"] = idx
    # the new tokens lie on the last page (all of them with last >= t): each sees every token of the other pages
    keys, values = (c["cache"][idx[:-1].long(), i].reshape(-1, hkv, d).float() for i in (0, 1))
    rep = hq // hkv
    s = torch.einsum("thd,khd->thk", c["q"].float(), keys.repeat_interleave(rep, 1)) * c["scale"]
    ref = torch.einsum("thk,khd->thd", torch.softmax(s, -1), values.repeat_interleave(rep, 1))
    status = torch.zeros(1, dtype=torch.int32, device=dev)
    print(f"case bad last page d={d} pages={pages} split={split}", flush=True)
    got = _call(c, dev, split, c["scale"], status)
    torch.testing.assert_close(got.float(), ref.to(torch.bfloat16).float(), **TOL)
    assert int(status.item()) == 1


def test_layer_takes_a_workspace_without_the_splits(dev):
    """The verify layer runs in the buffers it cannot do without (the attention then unsplit), as with the full size."""
    g = torch.Generator().manual_seed(10)
    h, f, hq, hkv, d, b, t = 256, 512, 8, 2, 64, 2, 3
    w = {k: v.to(dev) for k, v in configs.attn_layer_weights(g, h, f, hq, hkv, d).items()}
    c = _dev(configs.verify_rows_case([700, 90], t, hq, hkv, d, 16, g), dev)
    x = torch.randn(b, t, h, generator=g).bfloat16().to(dev)
    cos = torch.ones(b, t, 16, dtype=torch.bfloat16, device=dev)
    ws = layer.attn_verify_workspace(b, t, h, hq, hkv, d, f, dev)
    splits = _lib.load().axk_paged_prefill_workspace_size(b, b * t, hq, hkv, d)
    assert splits > 0
    outs = []
    for n in (ws.numel(), ws.numel() - (splits + 255) // 256 * 256):
        outs.append(layer.attn_layer_verify(x, w, cos, torch.zeros_like(cos), c["cache"].clone(), c["indptr"],
                                            c["indices"], c["last_page_len"], c["loc"], hq, 32, workspace=ws[:n]))
    torch.testing.assert_close(outs[0].float(), outs[1].float(), rtol=5e-2, atol=0.0625)
    with pytest.raises(_lib.AxkError):
        layer.attn_layer_verify(x, w, cos, torch.zeros_like(cos), c["cache"], c["indptr"], c["indices"],
                                c["last_page_len"], c["loc"], hq, 32, workspace=ws[:n - 256])


def test_split_under_capture(dev):
    """The Python operator's scratch comes from the graph's pool under capture; every replay equals the eager call."""
    g = torch.Generator().manual_seed(11)
    c = _dev(configs.prefill_case([5], [2000], 16, 2, 128, 64, g), dev)
    out = torch.empty_like(c["q"])
    args = (c["q"], c["cache"], c["qo_indptr"], c["indptr"], c["indices"], c["last_page_len"])
    want = attention.paged_prefill(*args).cpu()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        attention.paged_prefill(*args, output=out)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        attention.paged_prefill(*args, output=out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.cpu().view(torch.int16), want.view(torch.int16))
        torch.randn(1 << 20, device=dev).sum().item()


@pytest.mark.parametrize("qlens,kv_lens,split", [([4] * 8, [100] * 8, False), ([4], [320], False), ([4], [448], True),
                                                 ([4] * 8, [320] * 7 + [448], True)])
def test_short_sequences_are_not_split(dev, monkeypatch, qlens, kv_lens, split):
    """The operator splits by the cached tokens a sequence has room for, not by their sum."""
    c = _dev(configs.prefill_case(qlens, kv_lens, 16, 2, 128, 64, torch.Generator().manual_seed(3)), dev)
    names, call = [], _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *args: (names.append(name), call(name, *args))[1])
    got = attention.paged_prefill(c["q"], c["cache"], c["qo_indptr"], c["indptr"], c["indices"], c["last_page_len"])
    assert names == ["axk_paged_prefill_split" if split else "axk_paged_prefill"]
    ref = pa.paged_prefill(*(c[n].cpu() for n in ("q", "cache", "qo_indptr", "indptr", "indices", "last_page_len")),
                           c["scale"])
    torch.testing.assert_close(got.float().cpu(), ref.to(torch.bfloat16).float(), **TOL)


def test_workspace_of_the_caller(dev, monkeypatch):
    """A kept workspace takes the place of the call's own scratch, bit for bit, and nothing is allocated; without the memory
    for a scratch, or with a smaller workspace, the call runs unsplit."""
    c = _dev(configs.prefill_case([4, 3], [900, 1500], 16, 2, 128, 64, torch.Generator().manual_seed(4)), dev)
    args = (c["q"], c["cache"], c["qo_indptr"], c["indptr"], c["indices"], c["last_page_len"])
    want = attention.paged_prefill(*args)
    ws = attention.paged_prefill_workspace(2, 7, 16, 2, 128, dev)
    assert ws.numel() > 0 and attention.paged_prefill_workspace(2, 4096, 16, 2, 128, dev).numel() == 0
    out = torch.empty_like(want)
    before = torch.cuda.memory_stats(dev)["allocation.all.allocated"]
    attention.paged_prefill(*args, output=out, workspace=ws)
    assert torch.cuda.memory_stats(dev)["allocation.all.allocated"] == before
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
    whole = _call(c, dev, False, c["scale"]).to(dev)
    attention.paged_prefill(*args, output=out, workspace=ws[:-1])
    assert torch.equal(out.view(torch.int16), whole.view(torch.int16))

    def no_memory(*args, **kw):
        raise torch.OutOfMemoryError()

    out.zero_()
    with monkeypatch.context() as m:
        m.setattr(torch, "empty", no_memory)
        attention.paged_prefill(*args, output=out)
    assert torch.equal(out.view(torch.int16), whole.view(torch.int16))
    with pytest.raises(ValueError):
        attention.paged_prefill(*args, workspace=ws.view(torch.int32) if ws.numel() % 4 == 0 else ws[::2])
