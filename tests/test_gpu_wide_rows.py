"""fp32 activations above 4 tokens, per element: rows whose small values outlive their large ones, and single values.

The bars are relative to sum|x W| alone.  A row of a wide range beside weights that are zero at its large values
(the origin's atoms; int8 zeros) has outputs made of its small values only, which an error relative to the row's
largest value would swamp.
"""

import pytest
import torch

from oracle import torch_ref
from pollux_amd import castor
from pollux_amd.packed import (dequant_linear, dequant_linear_multi, dequantize_h24, h24_plane_layout, int8_linear,
                               int8_linear_argmax)

pytestmark = pytest.mark.gpu

KINDS = ["outlier", "deep", "mixed", "ladder", "pair"]


def _weight(dev, rows, cols, seed):
    """Packed weight: the origin's atom first in the odd rows, everywhere but first in every seventh row."""
    g = torch.Generator(device=dev).manual_seed(seed)
    idx = torch.randint(1, 196561, (rows, cols // 24), generator=g, device=dev)
    idx[1::2, :1] = 0
    idx[::7, :1] = torch.randint(1, 196561, (len(idx[::7]), 1), generator=g, device=dev)
    idx[::7, 1:] = 0
    sg = (torch.rand(rows, generator=g, device=dev) * 0.045 + 0.005).half()
    return castor.pack_indices(idx.reshape(-1)), sg


def _rows(dev, m, cols, kind, seed):
    """Activations with wide rows among ordinary ones; which rows are wide."""
    g = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn(m, cols, generator=g, device=dev)
    wide = torch.zeros(m, dtype=torch.bool, device=dev)
    wide[::3] = True
    wide[m - 1] = True
    n = int(wide.sum())
    if kind == "outlier":     # one large value, the rest a factor 2^-60 below
        x[wide] *= 2.0 ** -60
        x[wide, 0] = 1.0
    elif kind == "deep":      # the large values near fp32's top, the small ones far down
        x[wide] *= 1e-30
        x[wide, :24] *= 1e35
    elif kind == "mixed":     # every value its own power of two
        x[wide] *= torch.exp2(torch.randint(-70, 30, (n, cols), generator=g, device=dev).float())
    elif kind == "pair":      # two small values in the first atom, nothing else there
        x[wide, :24] = 0
        x[wide, 3], x[wide, 17] = 3e-20, -7e-25
    else:                     # just past what two fp16 parts hold: 2^-29 to 2^-27 of the largest
        x[wide] = (1 + torch.rand(n, cols, generator=g, device=dev)) * 2.0 ** -14
        x[wide, 0] = torch.exp2(13.0 + torch.rand(n, generator=g, device=dev) * 2)
    return x, wide


def _bar(x, w, cols, extra=0):
    # x's last bit, a rounding (2^-23: the MFMA cuts off) per MFMA of a step of 32 columns and of the final sums
    return (2.0 ** -23 + (6 * ((cols + 31) // 32) / 4 + 12 + extra) * 2.0 ** -23) * (x.abs() @ w.abs().T) + 1e-44


# both sides of every token tile (16, 32, 64), slab and large-batch edge; K with and without a whole last quad, K split
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("rows,cols,m", [
    (33, 120, 5), (48, 96, 16), (130, 960, 17), (64, 1920, 33), (257, 480, 64), (61, 2424, 65), (160, 7680, 70),
    (1921, 984, 200), (24, 9624, 321), (300, 480, 321), (130, 7680, 330), (1920, 1920, 400), (2000, 336, 513)])
def test_wide_rows(dev, rows, cols, m, kind):
    pk, sg = _weight(dev, rows, cols, rows + cols)
    x, wide = _rows(dev, m, cols, kind, m)
    w = dequantize_h24(pk, sg, rows, cols).double()
    bar = _bar(x.double(), w, cols)
    ref = x.double() @ w.T
    y = dequant_linear(pk, sg, rows, cols, x)
    worst = ((y.double() - ref).abs() / bar).max().item()
    print(f"[wide] {rows}x{cols} m={m} {kind}: {worst:.3f} of the bar", flush=True)
    assert worst <= 1.0
    assert torch.equal(y, dequant_linear(pk, sg, rows, cols, x, planes=h24_plane_layout(pk, rows * cols // 24)))
    # the ordinary rows beside them: the bits they have without them
    calm = x.clone()
    calm[wide] = 1.0
    assert torch.equal(y[~wide], dequant_linear(pk, sg, rows, cols, calm)[~wide])


# the norm fused into the copy, a row in 2, 4 and 8 registers a lane; not fused
@pytest.mark.parametrize("cols,m", [(480, 20), (504, 33), (960, 12), (960, 330), (984, 70), (2016, 40), (2400, 40), (2400, 330)])
def test_wide_rows_with_norm_and_epilogues(dev, cols, m):
    shapes = (130, 961)
    ws = [_weight(dev, r, cols, r) for r in shapes]
    x, _ = _rows(dev, m, cols, "outlier", m)
    g = torch.Generator(device=dev).manual_seed(1)
    nw = 1 + 0.1 * torch.randn(cols, generator=g, device=dev)
    res = [torch.randn(m, r, generator=g, device=dev) * 2.0 ** -60 for r in shapes]
    ys = dequant_linear_multi([(*w, r) for w, r in zip(ws, shapes)], cols, x, residuals=res, norm=(nw, 1e-8))
    n = x.double() * torch.rsqrt(x.double().square().mean(1, keepdim=True) + 1e-8) * nw.double()
    for (pk, sg), r, rs, y in zip(ws, shapes, res, ys):
        w = dequantize_h24(pk, sg, r, cols).double()
        # (the norm: half of its 11 + cols / 64 roundings of squares, root, quotient, two products)
        bar = _bar(n, w, cols, (11 + cols // 64) // 2 + 5) + 2.0 ** -23 * (rs.double().abs() + (n @ w.T).abs())
        assert ((y.double() - (n @ w.T + rs.double())).abs() <= bar).all()


def test_wide_rows_without_finite_large_values(dev):
    # an infinite or NaN value beside small ones: its own token's outputs alone
    pk, sg = _weight(dev, 64, 480, 9)
    for m in (7, 330):
        x, wide = _rows(dev, m, 480, "outlier", m)
        x[0, 3], x[3, 5] = float("inf"), float("nan")
        y = dequant_linear(pk, sg, 64, 480, x)
        keep = torch.ones(m, dtype=torch.bool, device=dev)
        keep[[0, 3]] = False
        w = dequantize_h24(pk, sg, 64, 480).double()
        assert ((y.double() - x.double() @ w.T).abs()[keep] <= _bar(x.double(), w, 480)[keep]).all()
        assert torch.isnan(y[3]).all() and not torch.isfinite(y[0]).any()


# one value a row: the only errors are the last bit of x (2^-23) and of one sum (2^-23)
@pytest.mark.parametrize("rows,cols,m", [(64, 96, 5), (64, 480, 30), (130, 1920, 64), (130, 1920, 200), (640, 1920, 400)])
def test_single_values(dev, rows, cols, m):
    pk, sg = _weight(dev, rows, cols, 2)
    g = torch.Generator(device=dev).manual_seed(m)
    x = torch.zeros(m, cols, device=dev)
    at = torch.randint(0, cols, (m, 1), generator=g, device=dev)
    x.scatter_(1, at, torch.randn(m, 1, generator=g, device=dev))
    w = dequantize_h24(pk, sg, rows, cols).double()
    ref = x.double() @ w.T
    y = dequant_linear(pk, sg, rows, cols, x).double()
    print(f"[single] {rows}x{cols} m={m}: {((y - ref).abs() / ref.abs().clamp_min(1e-30)).max().item() * 2 ** 23:.3f} "
          "of 2^-23", flush=True)
    assert ((y - ref).abs() <= 2.0 ** -22 * ref.abs()).all()


def _int8(dev, rows, cols, seed):
    g = torch.Generator().manual_seed(seed)
    q = torch.randint(-127, 128, (rows, cols), dtype=torch.int8, generator=g)
    q[1::2, :24] = 0
    q[::7, 24:] = 0
    mu = (torch.rand(rows, generator=g) * 0.1 + 0.01).half()
    return q.to(dev), mu.to(dev), torch_ref.int8_materialize(q, mu).double().to(dev)


# x split once per call (these sizes' form) at 1, 2 and 4 token tiles, partial slabs, fused and unfused norm
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("normed", [False, True])
@pytest.mark.parametrize("rows,cols,m", [(130, 4096, 5), (520, 1920, 32), (130, 960, 65), (77, 2032, 40), (33_000, 112, 130)])
def test_int8_wide_rows(dev, rows, cols, m, kind, normed):
    if normed and kind == "deep":
        pytest.skip("its squares leave fp32")
    q, mu, w = _int8(dev, rows, cols, rows + m)
    x, wide = _rows(dev, m, cols, kind, m)
    g = torch.Generator(device=dev).manual_seed(1)
    nw = 1 + 0.1 * torch.randn(cols, generator=g, device=dev)
    norm, n = None, x.double()
    if normed:
        norm, n = (nw, 1e-8), n * torch.rsqrt(n.square().mean(1, keepdim=True) + 1e-8) * nw.double()
    y = int8_linear(q, mu, x, norm=norm)
    bar = _bar(n, w, cols, (11 + cols // 64) // 2 + 5 if normed else 0)
    worst = ((y.double() - n @ w.T).abs() / bar).max().item()
    print(f"[wide int8] {rows}x{cols} m={m} {kind} norm={normed}: {worst:.3f} of the bar", flush=True)
    assert worst <= 1.0
    ids = torch.empty(m, dtype=torch.long, device=dev)
    ya = int8_linear_argmax(q, mu, x, ids, norm=norm)
    assert torch.equal(ya, y) and torch.equal(ids, torch.argmax(y, -1))
    calm = x.clone()
    calm[wide] = 1.0
    assert torch.equal(y[~wide], int8_linear(q, mu, calm, norm=norm)[~wide])


@pytest.mark.parametrize("m", [5, 40, 200])
def test_int8_single_values(dev, m):
    q, mu, w = _int8(dev, 600, 1920, m)
    g = torch.Generator(device=dev).manual_seed(m)
    x = torch.zeros(m, 1920, device=dev)
    x.scatter_(1, torch.randint(0, 1920, (m, 1), generator=g, device=dev), torch.randn(m, 1, generator=g, device=dev))
    ref = x.double() @ w.T
    assert ((int8_linear(q, mu, x).double() - ref).abs() <= 2.0 ** -22 * ref.abs()).all()
