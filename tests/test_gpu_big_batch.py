"""The dequant-linear of large fp32 batches: which calls decode their weights into a copy first, and what that does.

A call that does sums in another order than one of up to 320 tokens, so its bits tell which it was.
"""

import pytest
import torch

from pollux_amd import castor
from pollux_amd.packed import dequant_linear, dequantize_h24

pytestmark = pytest.mark.gpu


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
