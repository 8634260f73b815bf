"""NN-T and NN-P on atoms near fp32's largest values and with NaN, against every code's exact score in float64.

Expected: the lowest row of the highest score; under NN-T the scores are fp32, so all that overflow tie.  An atom
whose runner-up lies within 24 * 2^-24 * 2 (|x|_2 |c|_2) of the best may differ (the bound on two fp32 sums).
"""

import pytest
import torch

from oracle import codebook as cb
from pollux_amd import castor

pytestmark = pytest.mark.gpu


def _expected(x, mode):
    c = torch.from_numpy(cb.codebook_f32()[1:]).to(x.device)
    a, c = (x.bfloat16().double(), c.bfloat16().double()) if mode == "fp32" else (x.double(), c.double())
    s = a @ c.T
    edge = torch.zeros(len(x), dtype=torch.bool, device=x.device)
    if mode == "fp32":
        edge = ((s - 2.0 ** 128).abs() <= 2.0 ** 106).any(1)  # (rounds up to infinity, or not)
        s = torch.where(s.float().isinf() & (s > 0), torch.full_like(s, 2.0 ** 128), s)
    best = s.max(1, keepdim=True).values
    tol = torch.where(best >= 2.0 ** 128, 0.0, 24 * 2.0 ** -24 * 2.0 * 2.01 * a.norm(dim=1, keepdim=True))
    near = ((s >= best - tol).sum(1) > 1) & (tol[:, 0] > 0)
    return (s == best).int().argmax(1) + 1, near | edge


def _atoms(dev, n, scale):
    g = torch.Generator(device=dev).manual_seed(7)
    return (torch.randn(n, 24, generator=g, device=dev).clamp(-3.3, 3.3) * scale)


# sums of |x| up to the scorers' limit (2^120, crossed by atoms of 5e34), past it, past fp32 (1.5e37), where the best
# scores overflow (1e38)
@pytest.mark.parametrize("mode", ["fp32", "pack"])
@pytest.mark.parametrize("scale", [2.0 ** 90, 1e33, 5e34, 7e34, 1e36, 1.5e37, 4e37, 1e38])
def test_huge_atoms(dev, mode, scale):
    x = _atoms(dev, 500, scale)
    got = castor.quantize_indices(x, mode=mode).long()
    want, near = _expected(x, mode)
    bad = (got != want) & ~near
    print(f"[huge] {mode} {scale:.1e}: {int(near.sum())} near, {int(bad.sum())} wrong", flush=True)
    assert near.float().mean() < 0.05 and not bad.any()


def test_huge_atoms_in_a_batch(dev):
    # the batched requantize under NN-T: a row scaled by its own size has coordinates of a few units
    g = torch.Generator(device=dev).manual_seed(3)
    mats = [torch.randn(r, 48, generator=g, device=dev) * s for r, s in ((40, 1.0), (30, 1e18), (50, 1e-3))]
    one = [castor.requantize_h24(w, mode="fp32") for w in mats]
    many = castor.requantize_h24_many(mats, mode="fp32")
    assert all(torch.equal(a["indices"], b["indices"]) for a, b in zip(one, many))


@pytest.mark.parametrize("mode", ["fp32", "pack"])
def test_blocks_of_nan_atoms(dev, mode):
    x = _atoms(dev, 5000, 1.0)
    ref = castor.quantize_indices(x, mode=mode)
    x[1000:4000, 11] = float("nan")
    x[1000:4000:2, 12] = float("inf")
    got = castor.quantize_indices(x, mode=mode)
    assert torch.equal(got[:1000], ref[:1000]) and torch.equal(got[4000:], ref[4000:]) and not got[1000:4000].any()


@pytest.mark.parametrize("n", [1, 2, 5, 24])
def test_infinite_coordinates_under_pack(dev, n):
    # the lowest row with x's sign at every infinite coordinate (its score is infinite; a zero there makes it NaN,
    # another sign NaN or -inf); the origin where there is none
    x = _atoms(dev, 700, 1.0)
    g = torch.Generator(device=dev).manual_seed(n)
    at = torch.rand(700, 24, generator=g, device=dev).argsort(1)[:, :n]
    sign = torch.randint(0, 2, (700, n), generator=g, device=dev).float() * 2 - 1
    x.scatter_(1, at, sign * float("inf"))
    x[500:, 0] = float("inf")
    want = []
    c = torch.from_numpy(cb.codebook_int8()[1:].copy()).to(dev).float()
    for a in x.split(50):
        s = torch.where(a.isinf(), a.sign(), torch.zeros_like(a))
        ok = (s @ c.sign().T) == a.isinf().sum(1, keepdim=True)
        want.append(torch.where(ok.any(1), ok.int().argmax(1) + 1, 0))
    assert torch.equal(castor.quantize_indices(x, mode="pack").long(), torch.cat(want))
