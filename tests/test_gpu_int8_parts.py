"""The INT8 head above 4 tokens against float64: both MFMA forms (x split once per call in a workspace; split by
every block without one), at the edges of their tiles and of the split's number ranges."""

import pytest
import torch

from oracle import torch_ref

pytestmark = pytest.mark.gpu

# x split once: one row and partial row blocks, 1, 2 and 4 token tiles, partial slabs, rows of parts of a double step
# of 64 columns, waves without a step (80 columns), the last row length whose norm is fused into the split (2,016) and
# the first that is not, the longest, the least work of the rule at each token count
ONCE = [(1, 1040, 33), (63, 624, 64), (130, 960, 65), (64, 4096, 5), (65, 2016, 16), (70, 2032, 17), (520, 1920, 32),
        (513, 2016, 40), (77, 2032, 40), (200, 4096, 129), (40_000, 80, 300), (33_000, 112, 130), (70, 608, 33)]
# split by every block: just below that work, and the smallest
BLOCK = [(1, 16, 5), (63, 48, 16), (65, 80, 32), (513, 112, 64), (70, 592, 33), (70, 1184, 32), (200, 1984, 16)]
SHAPES = [(*s, True) for s in ONCE] + [(*s, False) for s in BLOCK]


def _inputs(dev, rows, cols, m):
    g = torch.Generator().manual_seed(rows + 3 * cols + 7 * m)
    q = torch.randint(-128, 128, (rows, cols), dtype=torch.int8, generator=g)
    # row scales from fp16 subnormals (weights that round on the subnormal grid) to the largest without overflow
    mu = torch.pow(2.0, torch.rand(rows, generator=g) * 37.0 - 22.0).to(torch.float16)
    mu[0] = 0.05
    if rows > 8:
        mu[3], mu[5], mu[7] = 0.0, 1.3e-4, 6e4
        q[7].clamp_(min=-127)
    x = torch.randn(m, cols, generator=g)
    x[1] *= torch.pow(2.0, torch.rand(cols, generator=g) * 24.0 - 20.0)  # a wide range within one row
    x[2] *= 1e-30
    x[3] *= 1e20
    x[4] = 0.0
    return q.to(dev), mu.to(dev), x.to(dev)


def _direct(q, mu, x, norm):
    from pollux_amd import _lib

    y = torch.empty(x.shape[0], q.shape[0], device=x.device)
    nw, eps = norm if norm else (None, 0.0)
    st = _lib.lib().plx_int8_linear(_lib.ptr(q), _lib.ptr(mu), q.shape[0], q.shape[1], _lib.ptr(x), x.shape[0],
                                    _lib.ptr(nw), eps, _lib.ptr(y), _lib.stream_of(x.device))
    _lib.check(st, "plx_int8_linear")
    return y


@pytest.mark.parametrize("rows,cols,m,once", SHAPES)
@pytest.mark.parametrize("normed", [False, True])
def test_both_forms_against_float64(rows, cols, m, once, normed):
    from pollux_amd import _lib
    from pollux_amd.packed import int8_linear

    assert (_lib.lib().plx_int8_linear_workspace_bytes(rows, cols, m) > 0) == once

    dev = torch.device("cuda:0")
    q, mu, x = _inputs(dev, rows, cols, m)
    if normed:
        x[3] = x[0] * 1e6  # (the squares of 1e20 leave fp32)
    w = torch_ref.int8_materialize(q, mu).double().cpu()
    nw = 1.0 + 0.1 * torch.randn(cols, generator=torch.Generator().manual_seed(1))
    norm = (nw.to(dev), 1e-8) if normed else None
    xd = x.double().cpu()
    if normed:
        xd = xd * torch.rsqrt(xd.square().mean(-1, keepdim=True) + 1e-8) * nw.double()
    ref, scale = xd @ w.t(), xd.abs() @ w.abs().t()
    # fp32 roundings of a sum, each at most 2^-23 of sum|x||w| (the MFMA rounds down): six MFMAs (two for the split
    # x) of a wave's share of the steps of 32 columns, three additions over the waves, two scales, the split's last
    # bit of x; the norm: the sum of squares (half of its 11 + cols / 64 roundings), root, quotient, two products
    steps = 2 * ((cols + 255) // 256)
    for name, per_step, y in (("layer", 2 if once else 6, int8_linear(q, mu, x, norm=norm)),
                              ("no workspace", 6, _direct(q, mu, x, norm))):
        n = per_step * steps + 6 + ((11 + cols // 64) // 2 + 5 if normed else 0)
        err = (y.double().cpu() - ref).abs()
        bound = n * 2.0**-23 * scale + 2.0**-140  # (and the smallest fp32 values)
        print(f"[int8 parts] {rows}x{cols} m={m} norm={normed} {name}: err / bound {(err / bound).max():.2e}", flush=True)
        assert (err <= bound).all(), name


def test_split_once_inf_nan_and_argmax_route():
    from pollux_amd.packed import int8_linear, int8_linear_argmax

    dev = torch.device("cuda:0")
    q, mu, x = _inputs(dev, 200, 624, 70)
    x[10, 5], x[11, 6], mu[9] = float("inf"), float("nan"), float("nan")
    q[:, 5] = torch.where(q[:, 5] == 0, 1, q[:, 5])
    y = int8_linear(q, mu, x)
    w = torch_ref.int8_materialize(q, mu).float().cpu()
    ok = torch.ones(200, dtype=torch.bool)
    ok[9] = False
    assert torch.isnan(y[:, 9]).all() and torch.isnan(y[11]).all()
    live = ok & (w[:, 5] != 0)
    assert torch.equal(y[10].cpu()[live], float("inf") * torch.sign(w[live, 5]))
    fine = [i for i in range(70) if i not in (10, 11)]
    assert torch.isfinite(y[fine][:, ok.to(dev)]).all()
    # the argmax route's outputs are the same bits
    ids = torch.empty(70, dtype=torch.long, device=dev)
    ya = int8_linear_argmax(q, mu, x, ids)
    assert torch.equal(ya.view(torch.int32), y.view(torch.int32)) and torch.equal(ids, torch.argmax(y, -1))


def test_split_once_replays_from_a_graph():
    from pollux_amd.packed import int8_linear

    dev = torch.device("cuda:0")
    q, mu, x = _inputs(dev, 130, 2032, 20)
    norm = (torch.ones(2032, device=dev), 1e-8)
    x[3] = x[0]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        int8_linear(q, mu, x, norm=norm)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = int8_linear(q, mu, x, norm=norm)
    for _ in range(3):
        x.copy_(torch.randn_like(x))
        want = int8_linear(q, mu, x, norm=norm)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
