"""The batched dequant-linear (fp32 x as two scaled fp16 parts, bf16 x as it is) against float64.

Per element the bar is (2^-23 + (K / 32 + 42) 2^-24) sum|x W|: the last bit of x that the two parts may drop (rows
of too wide a range for them are three exact bf16 parts), and one fp32 rounding per 32-column step plus those inside
a step and of the final sums.
"""

import numpy as np
import pytest
import torch

from oracle import codebook as cb
from pollux_amd import castor
from pollux_amd.packed import dequant_linear, dequant_linear_multi, dequantize_h24, h24_plane_layout

pytestmark = pytest.mark.gpu


def _weight(dev, rows, cols, seed, sigma=None):
    g = torch.Generator(device=dev).manual_seed(seed)
    idx = torch.randint(0, 196561, (rows * cols // 24,), generator=g, device=dev)
    sg = (torch.rand(rows, generator=g, device=dev) * 0.045 + 0.005).half() if sigma is None else sigma
    return castor.pack_indices(idx), sg


def _bar(x, w, cols):
    return (2.0 ** -23 + (cols / 32 + 42) * 2.0 ** -24) * (x.abs() @ w.abs().T) + 1e-38


# rows and tokens around the tiles (16 tokens, 32 and 128 rows, 64- and 128-token blocks), K with and without a
# whole last quad of 96 columns, packed stream and plane layout
@pytest.mark.parametrize("planes", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,cols,m", [
    (32, 24, 5), (48, 96, 16), (33, 120, 17), (130, 480, 33), (257, 1920, 64), (127, 984, 65), (129, 1920, 128),
    (384, 504, 129), (1921, 960, 160), (1920, 1920, 192), (640, 7680, 200), (61, 2424, 257), (2000, 336, 513),
    (5760, 1920, 300), (1, 48, 300), (24, 9624, 200), (2000, 1920, 1024), (300, 7680, 384), (129, 120, 321), (24, 9624, 350)])
def test_against_float64(dev, rows, cols, m, dtype, planes):
    pk, sg = _weight(dev, rows, cols, rows + cols)
    g = torch.Generator(device=dev).manual_seed(m)
    x = torch.randn(m, cols, generator=g, device=dev).to(dtype)
    pl = h24_plane_layout(pk, rows * cols // 24) if planes else None
    y = dequant_linear(pk, sg, rows, cols, x, planes=pl)
    w = dequantize_h24(pk, sg, rows, cols).double()
    err = (y.double() - x.double() @ w.T).abs()
    worst = (err / _bar(x.double(), w, cols)).max().item()
    print(f"[batched] {rows}x{cols} m={m} {dtype}: worst {worst:.3f} of the bar, "
          f"rel {(err.norm() / (x.double() @ w.T).norm()).item():.2e}", flush=True)
    assert worst <= 1.0


@pytest.mark.parametrize("m", [7, 64, 200, 330])
@pytest.mark.parametrize("what", ["tiny", "huge", "outliers", "subnormal", "mixed"])
def test_activation_ranges(dev, m, what):
    rows, cols = 200, 960
    pk, sg = _weight(dev, rows, cols, 3)
    g = torch.Generator(device=dev).manual_seed(m)
    x = torch.randn(m, cols, generator=g, device=dev)
    if what == "tiny":
        x *= 1e-30
    elif what == "huge":
        x *= 1e30
    elif what == "outliers":
        x[:, 7::100] *= 1e6
    elif what == "subnormal":
        x *= 2.0 ** -140  # (a part of a value below 2^-126 has fewer bits: absolute bar)
    else:  # each row its own scale, columns over 2^40
        x *= torch.exp2(torch.randint(-60, 60, (m, 1), generator=g, device=dev).float())
        x *= torch.exp2(-torch.rand(m, cols, generator=g, device=dev) * 40)
    y = dequant_linear(pk, sg, rows, cols, x)
    w = dequantize_h24(pk, sg, rows, cols).double()
    xd = x.double()
    bar = _bar(xd, w, cols)
    if what == "subnormal":
        bar = bar + 2.0 ** -149 * cols
    assert ((y.double() - xd @ w.T).abs() <= bar).all()


@pytest.mark.parametrize("m", [7, 200, 330])
def test_row_scale_ranges(dev, m):
    # fp16 row scales from subnormal (weights of a few bits, or none) to where the largest weights overflow
    sg = torch.tensor([0.0, 6e-8, 1e-7, 3e-6, 1e-4, 1.0, 300.0, 40_000.0], device=dev).half().repeat(8)
    rows, cols = sg.numel(), 480
    pk, sg = _weight(dev, rows, cols, 4, sg)
    g = torch.Generator(device=dev).manual_seed(m)
    x = torch.randn(m, cols, generator=g, device=dev)
    w = dequantize_h24(pk, sg, rows, cols).double()
    y = dequant_linear(pk, sg, rows, cols, x).double()
    ref, fine = x.double() @ w.T, torch.isfinite(w).all(1)
    assert ((y - ref).abs() <= _bar(x.double(), w, cols))[:, fine].all()
    assert not torch.isfinite(y[:, ~fine]).any()


@pytest.mark.parametrize("m", [7, 200, 330])
def test_bad_tokens_stay_alone(dev, m):
    rows, cols = 160, 480
    pk, sg = _weight(dev, rows, cols, 5)
    g = torch.Generator(device=dev).manual_seed(m)
    x = torch.randn(m, cols, generator=g, device=dev)
    ref = dequant_linear(pk, sg, rows, cols, x)
    x[1, 5], x[3, 9] = float("nan"), float("inf")
    y = dequant_linear(pk, sg, rows, cols, x)
    keep = torch.ones(m, dtype=torch.bool, device=dev)
    keep[[1, 3]] = False
    assert torch.equal(y[keep], ref[keep]) and not torch.isfinite(y[[1, 3]]).any()


@pytest.mark.parametrize("m", [16, 150, 330])
def test_epilogues_and_targets(dev, m):
    # the norm prologue, GELU and residuals over several weights: the same as separate calls
    cols, shapes = 960, (130, 960, 64)
    ws = [_weight(dev, r, cols, r) for r in shapes]
    g = torch.Generator(device=dev).manual_seed(m)
    x = torch.randn(m, cols, generator=g, device=dev)
    nw = 1 + 0.1 * torch.randn(cols, generator=g, device=dev)
    res = [torch.randn(m, r, generator=g, device=dev) for r in shapes]
    ys = dequant_linear_multi([(*w, r) for w, r in zip(ws, shapes)], cols, x, residuals=res, gelu=True, norm=(nw, 1e-8))
    n = x.double() * torch.rsqrt(x.double().square().mean(1, keepdim=True) + 1e-8) * nw.double()
    for (pk, sg), r, rs, y in zip(ws, shapes, res, ys):
        w = dequantize_h24(pk, sg, r, cols).double()
        z = n @ w.T
        ref = torch.nn.functional.gelu(z) + rs.double()
        assert ((y.double() - ref).abs() <= 2 * _bar(n, w, cols) + 2.0 ** -22 * (z.abs() + rs.abs().double())).all()
