"""The dequant-linear of large fp32 batches: which calls decode their weights into a copy first, and what that does.

A call that does sums in another order than one of up to 320 tokens, so its bits tell which it was.
"""

import pytest
import torch

from pollux_amd import _lib, castor
from pollux_amd.packed import dequant_linear, dequant_linear_multi, dequantize_h24, int8_linear

pytestmark = pytest.mark.gpu
X_F32 = 1


def _weight(dev, rows, cols, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    idx = torch.randint(0, 196561, (rows * cols // 24,), generator=g, device=dev)
    return castor.pack_indices(idx), (torch.rand(rows, generator=g, device=dev) * 0.045 + 0.005).half()


def _bar(x, w, cols):
    return (2.0 ** -23 + (cols / 32 + 42) * 2.0 ** -24) * (x.abs() @ w.abs().T) + 1e-38


def _in_small_batches(pk, sg, rows, cols, x):
    return torch.cat([dequant_linear(pk, sg, rows, cols, part) for part in x.split(256)])


# one call on either side of each edge: tokens, products, columns
@pytest.mark.parametrize("rows,cols,m,big", [
    (1920, 1920, 320, False), (1920, 1920, 321, True), (1250, 96, 1000, True), (1249, 96, 1000, False),
    (624, 480, 400, False), (625, 480, 400, True), (24, 1920, 1024, False)])
def test_both_sides_of_the_rule(dev, rows, cols, m, big):
    pk, sg = _weight(dev, rows, cols, rows)
    x = torch.randn(m, cols, generator=torch.Generator(device=dev).manual_seed(m), device=dev)
    w = dequantize_h24(pk, sg, rows, cols).double()
    y = dequant_linear(pk, sg, rows, cols, x)
    assert torch.equal(y, _in_small_batches(pk, sg, rows, cols, x)) != big
    assert ((y.double() - x.double() @ w.T).abs() <= _bar(x.double(), w, cols)).all()


def _call(pk, sg, rows, cols, x, ws, nbytes):
    y = torch.empty(x.shape[0], rows, device=x.device)
    st = _lib.lib().plx_dequant_linear(_lib.ptr(pk), pk.numel(), _lib.ptr(sg), rows, cols, _lib.ptr(x), X_F32, x.shape[0],
                                       _lib.ptr(y), _lib.ptr(ws), nbytes, _lib.stream_of(x.device))
    return st, y


# a buffer sized once for the largest batch of a program serves the smaller ones; room for nothing but the sums that
# the kernel of small batches splits is enough, less is refused
@pytest.mark.parametrize("rows,cols,top", [(1920, 1920, 4000), (700, 7680, 2048), (7680, 480, 1500)])
def test_smaller_workspaces(dev, rows, cols, top):
    pk, sg = _weight(dev, rows, cols, 1)
    w = dequantize_h24(pk, sg, rows, cols).double()
    size = _lib.lib().plx_dequant_linear_workspace_bytes
    full = size(rows, cols, top, X_F32)
    ws = torch.empty(full, dtype=torch.uint8, device=dev)
    for m in (5, 64, 320, 321, 500, 1000):
        x = torch.randn(m, cols, generator=torch.Generator(device=dev).manual_seed(m), device=dev)
        ref = x.double() @ w.T
        head = (m + 63) // 64 * ((cols + 95) // 96 * 3 * 12288 + 256)
        slab = size(rows, cols, 64, X_F32) - ((cols + 95) // 96 * 3 * 12288 + 256)  # the partials of a slab
        least = head + (m + 63) // 64 * slab
        copy = (rows + 127) // 128 * 128 * ((cols + 95) // 96 * 192 + 4)  # (one chunk)
        for n in (full, size(rows, cols, m, X_F32), max(least, head + copy), least):
            st, y = _call(pk, sg, rows, cols, x, ws, min(n, full))
            _lib.check(st, "plx_dequant_linear")
            assert ((y.double() - ref).abs() <= _bar(x.double(), w, cols)).all(), (m, n)
        assert _call(pk, sg, rows, cols, x, ws, least - 1)[0] != 0


@pytest.mark.parametrize("rows,cols,m", [(50_688, 1920, 16), (130, 4096, 70)])
def test_argmax_with_room_for_the_keys_alone(dev, rows, cols, m):
    g = torch.Generator(device=dev).manual_seed(m)
    q = torch.randint(-127, 128, (rows, cols), generator=g, device=dev, dtype=torch.int8)
    mu = (torch.rand(rows, generator=g, device=dev) * 0.1 + 0.01).half()
    x = torch.randn(m, cols, generator=g, device=dev)
    keys = 8 * m * ((rows + 63) // 64)
    ws = torch.empty(keys, dtype=torch.uint8, device=dev)
    y, ids = torch.empty(m, rows, device=dev), torch.empty(m, dtype=torch.long, device=dev)

    def call(n):
        return _lib.lib().plx_int8_linear_argmax(_lib.ptr(q), _lib.ptr(mu), rows, cols, _lib.ptr(x), m, None, 0.0,
                                                 _lib.ptr(y), _lib.ptr(ids), None, 0, None, _lib.ptr(ws), n,
                                                 _lib.stream_of(dev))

    assert call(keys - 1) != 0
    _lib.check(call(keys), "plx_int8_linear_argmax")
    assert torch.equal(ids, torch.argmax(y, -1))
    ref = int8_linear(q, mu, x)
    assert (y - ref).norm() <= 1e-6 * ref.norm()


def _splits(rows, cols, m):
    """The plan's chunks of rows and K splits (bg_plan)."""
    nq, blocks = (cols + 95) // 96, (rows + 127) // 128
    fit = max(1, (24 << 20) // (nq * 96) // 128)
    chunks = (blocks + fit - 1) // fit
    per, steps, best = (blocks + chunks - 1) // chunks, 3 * nq, None
    for sp in range(1, max(1, min(16, steps // 8)) + 1):
        each = (steps + sp - 1) // sp + 1 & ~1
        cost = (per * ((m + 127) // 128) * sp + 511) // 512 * each + (
            3.0 + (2 * sp + 1) * (m * rows) * 1e-6 / chunks if sp > 1 else 0.0)
        if best is None or cost < best[0]:
            best = cost, (steps + each - 1) // each
    return chunks, best[1]


# several chunks of decoded rows (the last with a partial block), with and without K splits; residuals added by the
# GEMM itself (no K split: vector stores, and scalar ones for rows no multiple of 4) and by the split sum; GELU
@pytest.mark.parametrize("rows,cols,m,chunks,split", [
    (16_500, 1920, 330, 2, True), (16_500, 1920, 1100, 2, False), (33_333, 960, 400, 2, False), (640, 480, 400, 1, False),
    (641, 480, 400, 1, False), (1283, 336, 321, 1, False), (1283, 1920, 321, 1, True), (960, 960, 330, 1, True)])
@pytest.mark.parametrize("gelu", [False, True])
def test_chunks_and_epilogues(dev, rows, cols, m, chunks, split, gelu):
    n, splits = _splits(rows, cols, m)
    assert n == chunks and (splits > 1) == split
    pk, sg = _weight(dev, rows, cols, rows)
    g = torch.Generator(device=dev).manual_seed(m)
    x, res = torch.randn(m, cols, generator=g, device=dev), torch.randn(m, rows, generator=g, device=dev)
    w = dequantize_h24(pk, sg, rows, cols).double()
    z = x.double() @ w.T
    bar = _bar(x.double(), w, cols)
    del w
    for r in (None, res):
        y, = dequant_linear_multi([(pk, sg, rows)], cols, x, residuals=[r], gelu=gelu)
        ref = torch.nn.functional.gelu(z) if gelu else z
        ref = ref if r is None else ref + r.double()
        # (GELU's slope is below 1.13; its own fp32 steps and the residual's sum: 2^-22 of their size)
        tol = 1.13 * bar + 2.0 ** -22 * (z.abs() + res.double().abs())
        assert ((y.double() - ref).abs() <= tol).all()
