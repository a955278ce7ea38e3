"""GPU parity of the MoE decode kernels above 64 tokens, where the activation rows per pass (8, 12 or 16) follow the rows an
expert has: experts of one pass and of several, at the rows where the choice changes, with and without a shared expert of
another width, and the unstaged kernels (widths that are not whole batches, or more than 8 rows an expert). Bars of
tests/test_gpu_moe.py."""
import pytest
import torch

from axk import configs
from test_gpu_moe import _check_layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,h,e,f,fs,k", [
    (65, 512, 33, 256, 256, 4),    # just below 8 rows an expert: gate-up 12, down 16
    (65, 512, 32, 256, 256, 4),    # just above 8: unstaged, 16 rows
    (65, 512, 64, 256, 512, 4),    # 4 rows: gate-up 8, down 8; a wider shared expert
    (80, 256, 64, 512, 256, 4),    # 5 rows: gate-up 8, down 16
    (81, 256, 64, 512, 0, 4),      # past 5: gate-up 12; no shared expert
    (256, 256, 8, 256, 256, 2),    # 64 rows an expert: unstaged, several passes of each
    (200, 512, 300, 256, 256, 2),  # 1.3 rows: single passes, more than 256 experts
    (100, 512, 16, 96, 160, 3),    # staged gate-up, unstaged down
    (100, 384, 16, 256, 256, 3),   # unstaged gate-up, staged down
])
def test_rows_per_pass(dev, t, h, e, f, fs, k):
    g = torch.Generator().manual_seed(t + h + e)
    w = configs.moe_weights(g, hidden=h, experts=e, inter=f, shared_inter=max(fs, 32), router_std=0.5)
    if fs == 0:
        for n in ("w_gate", "s_gate", "w_up", "s_up", "w_down", "s_down", "w_shg"):
            w.pop(n)
    c = {"h2": torch.randn(t, h, generator=g).to(torch.bfloat16),
         "x_res": torch.randn(t, h, generator=g).to(torch.bfloat16), "weights": w, "top_k": k}
    print(f"case t={t} h={h} e={e} f={f} fs={fs} k={k}", flush=True)
    _check_layer(c, dev)


@pytest.mark.parametrize("t,h,e,f,fs,k", [
    (257, 256, 64, 128, 128, 2),   # 8 rows an expert: 32-row tiles
    (260, 256, 20, 128, 128, 2),   # 26 rows: 32-row tiles, some experts over one
    (280, 256, 20, 64, 64, 2),     # past 26 (28): 64-row tiles, widths without whole scale dwords
    (280, 256, 10, 192, 0, 2),     # 56 rows: the last of the 64-row tiles, no shared expert
    (300, 192, 10, 128, 128, 2),   # past 56: 128-row tiles
    (305, 256, 5, 128, 128, 2),    # 122 rows: 160-row tiles
    (330, 128, 4, 192, 64, 2),     # 165 rows: 160-row tiles, most experts over one
    (340, 256, 4, 128, 128, 2),    # 170: 128-row tiles again
    (300, 256, 2, 128, 128, 1),    # one expert near 150, top-1
    (300, 128, 40, 1152, 64, 2),   # 15 rows, a long down reduction: 128-row tiles
    (300, 192, 40, 128, 128, 2),   # 15 rows, no whole scale dwords: 64-row tiles
    (280, 192, 10, 1152, 0, 2),    # 56 rows of both kinds: 64-row tiles
    (280, 4096, 14, 64, 64, 2),    # 40 rows: from hidden 4096 on the last of the 64-row tiles
    (290, 4096, 14, 128, 0, 2),    # past 40: 128-row tiles
    (272, 4096, 4, 64, 64, 2),     # 136 rows: the last of the 128-row tiles there
    (280, 4096, 4, 64, 64, 2),     # past 136: 160-row tiles
    (304, 4096, 4, 64, 0, 2),      # 152: the last of them
])
def test_prefill_tile_rows(dev, t, h, e, f, fs, k):
    test_rows_per_pass(dev, t, h, e, f, fs, k)
