"""GPU parity of the runtime-weight linears at 17 .. 127 rows of wide matrices, where the dense GEMM takes over from the
group kernel: both sides of each threshold with the tile of 32 rows, the tiles of 64 and 128 rows (which need 256 workgroups)
at their edges in each epilogue, ragged channel counts, and a decode layer whose MLP takes the SwiGLU form. Bars as
tests/test_gpu_linear_prefill.py."""
import pytest
import torch

import axk
from axk import configs, layer
from oracle import layer as olayer
from oracle import mx
from test_gpu_linear_prefill import _close

pytestmark = pytest.mark.gpu
FUSED_TOL = dict(rtol=5e-2, atol=0.0625)


def _run(fmt, m, n, k, out_dtype, dev):
    g = torch.Generator().manual_seed(m * 7 + n + k)
    a = torch.randn(m, k, generator=g).to(torch.bfloat16)
    bias = torch.randn(n, generator=g) / 8
    rb = bias.to(out_dtype).float()
    kw = dict(out_dtype=out_dtype, bias=bias.to(dev))
    if fmt == "mxfp4":
        w, s = configs.mxfp4_weight(n, k, g)
        return a, axk.mxfp4_gemm(a.to(dev), w.to(dev), s.to(dev), **kw), rb, mx.dequant_mxfp4(w.numpy(), s.numpy())
    if fmt == "nvfp4":
        w = configs.pack_codes(torch.randint(0, 16, (n, k), generator=g, dtype=torch.uint8))
        s = torch.randint(0x28, 0x38, (n, k // 16), generator=g, dtype=torch.uint8)
        got = axk.nvfp4_gemm(a.to(dev), w.to(dev), s.to(dev), torch.tensor([0.05], device=dev), **kw)
        return a, got, rb, mx.dequant_nvfp4(w.numpy(), s.numpy(), 0.05)
    if fmt == "fp8":
        w, s = configs.fp8_proj_weight(n, k, g)
        got = axk.fp8_gemm(a.to(dev), w.to(dev), None, s.to(dev), **kw)
        return a, got, rb, mx.e4m3_table()[w.numpy()] * s.numpy()[:, None]
    codes = torch.randint(0, 0x7B, (n, k), generator=g, dtype=torch.uint8)  # finite in both formats
    s = torch.randint(119, 124, (n, k // 32), generator=g, dtype=torch.uint8)
    if fmt == "e5m2":
        codes = codes & 0x43  # magnitudes up to 3.5
    return a, axk.mxfp8_gemm(a.to(dev), codes.to(dev), s.to(dev), fmt=fmt, **kw), rb, mx.dequant_mxfp8(
        codes.numpy(), s.numpy(), fmt)


@pytest.mark.parametrize("fmt", ["mxfp4", "nvfp4", "fp8", "e4m3", "e5m2"])
@pytest.mark.parametrize("m,n,k", [(16, 8200, 256), (17, 24600, 256), (32, 24320, 128), (33, 8200, 256), (64, 7936, 128),
                                   (64, 16390, 384), (65, 8000, 256), (127, 8200, 128), (128, 300, 256),
                                   (40, 8200, 192)])
def test_rows_of_wide_matrices(dev, fmt, m, n, k):
    out_dtype = torch.float32 if m % 2 else torch.bfloat16
    if fmt != "fp8" and k % 128:
        k = 320  # a K of whole 64s but not of whole scale dwords (the group or the unstaged kernel)
    print(f"{fmt} m={m} n={n} k={k} {out_dtype}", flush=True)
    a, got, bias, w = _run(fmt, m, n, k, out_dtype, dev)
    wt = torch.from_numpy(w).float()
    _close(got, a.float() @ wt.T + bias, out_dtype, a, wt)


# Workgroups are ceil(n / 256) x ceil(m / rows), and the tile is the largest that gives 256 of them: 64 rows at (40, ..) and
# (1000, ..), 128 at the others in 4 bit (64 in 8 bit, which has no more).
@pytest.mark.parametrize("fmt", ["mxfp4", "nvfp4", "fp8", "e4m3"])
@pytest.mark.parametrize("m,n,k,out_dtype", [(40, 65550, 128, torch.bfloat16), (64, 65536, 128, torch.float32),
                                             (70, 65550, 128, torch.bfloat16), (130, 33000, 256, torch.float32),
                                             (1000, 4100, 256, torch.bfloat16), (2100, 4104, 256, torch.bfloat16)])
def test_tiles_of_64_and_128_rows(dev, fmt, m, n, k, out_dtype):
    print(f"{fmt} m={m} n={n} k={k} {out_dtype}", flush=True)
    a, got, bias, w = _run(fmt, m, n, k, out_dtype, dev)
    wt = torch.from_numpy(w).float()
    _close(got, a.float() @ wt.T + bias, out_dtype, a, wt)


# What the group kernel, which sums K in eight runs, is off the exact product by, and a tenth: 6.1e-8 of the norm, 8.0e-8
# where scale2 rounds once more, 1.21e-7 for codes of one sign.
RUN_ERROR = {"mxfp4": 6.7e-8, "nvfp4": 8.8e-8, "e4m3": 1.33e-7}


# Workgroups are ceil(n / 256) x ceil(m / rows), and the tile is the largest that gives 256 of them: 64 rows at (40, ..) and
# (1000, ..), 128 at the others in 4 bit (64 in 8 bit, which has no more).
@pytest.mark.parametrize("fmt", ["mxfp4", "nvfp4", "fp8", "e4m3"])
@pytest.mark.parametrize("m,n,k,out_dtype", [(40, 65550, 128, torch.bfloat16), (64, 65536, 128, torch.float32),
                                             (70, 65550, 128, torch.bfloat16), (130, 33000, 256, torch.float32),
                                             (1000, 4100, 256, torch.bfloat16), (2100, 4104, 256, torch.bfloat16)])
def test_tiles_of_64_and_128_rows(dev, fmt, m, n, k, out_dtype):
    print(f"{fmt} m={m} n={n} k={k} {out_dtype}", flush=True)
    a, got, bias, w = _run(fmt, m, n, k, out_dtype, dev)
    wt = torch.from_numpy(w).float()
    _close(got, a.float() @ wt.T + bias, out_dtype, a, wt)


# What the group kernel, which sums K in eight runs, is off the exact product by, and a tenth: 6.1e-8 of the norm, 8.0e-8
# where scale2 rounds once more, 1.21e-7 for codes of one sign (in six runs of uneven length: 1.36e-7).
RUN_ERROR = {"mxfp4": 6.7e-8, "nvfp4": 8.8e-8, "e4m3": 1.33e-7}


@pytest.mark.parametrize("fmt,m", [("mxfp4", 24), ("mxfp4", 100), ("nvfp4", 100), ("e4m3", 100)])
def test_fp32_rows_are_summed_in_runs(dev, fmt, m):
    """fp32 logits of an LM head's depth (K 2048) over 65536 channels are as near the exact product as the group kernel's,
    whatever tile the rows take (one chain over K: 8.1e-8, 1.25e-7 with scale2)."""
    a, got, bias, w = _run(fmt, m, 65536, 2048, torch.float32, dev)
    x, err, norm = a.double(), 0.0, 0.0
    for i in range(0, 65536, 8192):
        ref = x @ torch.from_numpy(w[i:i + 8192]).double().T + bias[i:i + 8192].double()
        err += float((got[:, i:i + 8192].cpu().double() - ref).square().sum())
        norm += float(ref.square().sum())
    print(f"{fmt} m={m} error {(err / norm) ** 0.5:.3g}", flush=True)
    assert (err / norm) ** 0.5 <= RUN_ERROR[fmt]


@pytest.mark.parametrize("mlp_fmt", ["mxfp4", "mxfp8"])
def test_layer_mlp_of_40_rows(dev, mlp_fmt):
    """40 sequences, MLP width 4096: gate | up take the dense GEMM's SwiGLU form, the other projections the group's."""
    g = torch.Generator().manual_seed(40)
    h, f, nk, nv, b = 256, 4096, 2, 4, 40
    w = configs.gdn_layer_weights(g, h, f, nk, nv, mlp_fmt=mlp_fmt)
    x = torch.randn(b, h, generator=g).bfloat16()
    st = torch.randn(b, nv, 128, 128, generator=g) * 0.02
    cv = torch.randn(b, 3, 2 * nk * 128 + nv * 128, generator=g).bfloat16()
    print(f"layer of 40 rows {mlp_fmt}", flush=True)
    out, _, _ = layer.gdn_layer_decode(x.to(dev), {n: t.to(dev) for n, t in w.items()}, st.to(dev), cv.to(dev), nk, nv,
                                       mlp_fmt=mlp_fmt)
    ref = olayer.gdn_layer_decode(x, w, st, cv, nk, nv, mlp_fmt=mlp_fmt)[0]
    torch.testing.assert_close(out.float().cpu(), ref.float(), **FUSED_TOL)


@pytest.mark.parametrize("fmt,b", [("mxfp4", 1100), ("mxfp4", 2039), ("nvfp4", 1100), ("nvfp4", 2039), ("mxfp8", 1100)])
def test_layer_tiles_of_64_and_128_rows(dev, fmt, b):
    """A decode layer of hidden and MLP width 4096 and 2048 over 1100 (tiles of 64 rows) or 2039 sequences (128 in 4 bit):
    the output projection, gate | up with SwiGLU, and down with the residual. The layer rounds to bf16 some ten times
    (2^-9 each, about 6e-3 of a row's norm if all fell differently): every row and column within 2e-2 of its norm, where
    16 wrong channels of a row are 6e-2."""
    g = torch.Generator().manual_seed(b)
    h, f, nk, nv = 4096, 2048, 1, 2
    w = configs.gdn_layer_weights(g, h, f, nk, nv, proj_fmt=fmt, mlp_fmt=fmt)
    x = torch.randn(b, h, generator=g).bfloat16()
    st = torch.randn(b, nv, 128, 128, generator=g) * 0.02
    cv = torch.randn(b, 3, 2 * nk * 128 + nv * 128, generator=g).bfloat16()
    print(f"layer of {b} rows {fmt}", flush=True)
    out, _, _ = layer.gdn_layer_decode(x.to(dev), {n: t.to(dev) for n, t in w.items()}, st.to(dev), cv.to(dev), nk, nv,
                                       proj_fmt=fmt, mlp_fmt=fmt)
    ref = olayer.gdn_layer_decode(x, w, st, cv, nk, nv, proj_fmt=fmt, mlp_fmt=fmt)[0].float()
    d = out.float().cpu() - ref
    for dim in (0, 1):
        assert (d.norm(dim=dim) <= 2e-2 * ref.norm(dim=dim)).all(), float((d.norm(dim=dim) / ref.norm(dim=dim)).max())
