"""A packed layer's bf16 outputs, rounded by the kernel that sums them, against its fp32 outputs rounded by torch."""

import pytest
import torch

from pollux_amd import _lib, castor
from pollux_amd.packed import PackedH24Linear, dequant_linear

pytestmark = pytest.mark.gpu


# one token from the plane layout (8, 32 and 64 lanes a row) and from the packed stream (rows past its 320 atoms);
# 2 tokens (the GEMV, no bf16 outputs of its own); the GEMM with and without a K split, rows in whole fours and
# not, 1, 2 and 4 token tiles, a partial second slab
@pytest.mark.parametrize("m", [1, 2, 3, 5, 17, 64, 65])
@pytest.mark.parametrize("rows,cols", [(24, 96), (25, 480), (1921, 1920), (5700, 480), (5701, 96), (30, 7704)])
@pytest.mark.parametrize("rounding", ["exact", "as_x"])
def test_bf16_outputs_equal_rounded_fp32(rows, cols, m, rounding):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(rows + cols + m)
    with torch.device(dev):
        layer = PackedH24Linear(cols, rows)
    layer.packed_weights.copy_(castor.pack_indices(
        torch.randint(0, 196_561, (layer.num_atoms,), generator=g, device=dev, dtype=torch.int32)))
    layer.sigma_rows.copy_((torch.rand(rows, generator=g, device=dev) * 0.05 + 0.005).half())
    layer.weight_rounding = rounding
    x = torch.randn(m, cols, generator=g, device=dev).bfloat16()
    x[-1, 3] = float("inf") if rounding == "exact" else 3e38  # infinities, NaN and overflow round as torch rounds them
    y = layer(x)
    planes = layer.plane_layout() if layer.use_plane_layout else None
    want = dequant_linear(layer.packed_weights, layer.sigma_rows, rows, cols, x, rounding, planes)
    assert want.dtype == torch.float32 and y.dtype == torch.bfloat16 and y.shape == want.shape
    want = want.to(torch.bfloat16)
    assert torch.equal(torch.isnan(y), torch.isnan(want))
    assert torch.equal(torch.nan_to_num(y, 7.0).view(torch.int16), torch.nan_to_num(want, 7.0).view(torch.int16))


def test_bf16_outputs_refused_where_no_kernel_writes_them():
    dev = torch.device("cuda:0")
    x = torch.zeros(8, 96, device=dev)
    pk, sg, y = torch.zeros(9 * 24, dtype=torch.uint8, device=dev), torch.ones(24, device=dev).half(), torch.zeros(8, 24, device=dev)
    for flags, m in ((32, 1), (32, 2), (32 | 1, 8), (32 | 4, 8)):  # the packed stream's GEMV, fp32 x, GELU
        st = _lib.lib().plx_dequant_linear(_lib.ptr(pk), pk.numel(), _lib.ptr(sg), 24, 96, _lib.ptr(x), flags, m,
                                           _lib.ptr(y), None, 0, _lib.stream_of(dev))
        with pytest.raises(ValueError, match="bf16 y"):
            _lib.check(st, "plx_dequant_linear")
