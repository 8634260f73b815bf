"""NN-T and NN-P through the structured scorers against every code's exact score in float64.

NN-T (castor.py:419-460): bf16 operands, the lowest code of the highest fp32 score.  NN-P (pack.py:167-177):
fp32 atoms and codebook.  Expected: the row of the highest float64 score; an atom whose runner-up lies
within 24 * 2^-24 * (|x|_2 |c|_2) * 2 of it (the bound on two fp32 sums of 24 terms, by Cauchy-Schwarz) may
differ, any other must agree.  Integer atoms have scores exact in every order, so the exact ties between codes
must be resolved alike on every atom -- also where a whole wave's lists overflow: among type-1/2 codes the one
whose antipodal pair lies in the earliest group of 256 pairs, then the lowest row; against a type-3 code (the
lowest of those that tie) the lower row.
"""

import numpy as np
import pytest
import torch

from oracle import codebook as cb
from pollux_amd import castor

pytestmark = pytest.mark.gpu

MODES = ["fp32", "pack"]
ORIGIN_T = float(np.float32(np.uint32(0x407FFFFF).view(np.float32))) / 2.0


def _operands(dev, x, mode):
    table = torch.from_numpy(cb.codebook_f32()).to(dev)
    if mode == "fp32":
        return x.bfloat16().double(), table.bfloat16().double()
    return x.double(), table.double()


def _tie_rank(dev):
    """Per row 1..: where it stands among tied codes of its family (lower wins), and whether it is a type-3 code."""
    nonzero = (cb.codebook_int8()[1:] != 0).sum(1)
    t3 = nonzero == 24
    rank = np.arange(196560, dtype=np.int64)
    pairs = np.flatnonzero(~t3)
    k = np.arange(len(pairs))
    rank[pairs] += np.minimum(k, len(pairs) - 1 - k) // 256 << 18
    return torch.from_numpy(rank).to(dev), torch.from_numpy(t3).to(dev)


def _expected(dev, x, mode):
    """(row of the best code, whether another code is within the fp32 sums' error of it) per atom."""
    idx, near = [], []
    rank, t3 = _tie_rank(dev)
    none = torch.full((), 1 << 40, device=dev)
    for part in x.split(512):
        a, c = _operands(dev, part, mode)
        s = a @ c[1:].T
        best, _ = s.max(1)
        hit = s == best[:, None]
        i = torch.minimum(*(torch.where(hit & fam, rank, none).min(1).values & (1 << 18) - 1 | has.logical_not().long() << 20
                            for fam, has in ((f, (hit & f).any(1)) for f in (t3, ~t3)))) + 1
        tol = 24 * 2.0 ** -24 * 2.0 * 2.01 * a.norm(dim=1)
        n = (s >= (best - tol)[:, None]).sum(1) > 1
        if mode == "fp32":
            i[best < ORIGIN_T] = 0
            n |= (best - ORIGIN_T).abs() <= tol
        else:
            i[a.norm(dim=1) < float(np.float32(1e-8))] = 0
        idx.append(i)
        near.append(n)
    return torch.cat(idx), torch.cat(near)


def _atoms(n, seed, dev):
    g = torch.Generator(device=dev).manual_seed(seed)
    return torch.randn(n, 24, generator=g, device=dev) * 2.0 ** 0.5


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("n", [1, 15, 63, 65, 257, 4097, 98_304, 131_071, 131_073])
def test_random_atoms_at_the_launch_sizes(dev, mode, n):
    # 1 atom tile per wave below 98,304 atoms, 2 below 131,072, else 4
    x = _atoms(n, n, dev)
    got = castor.quantize_indices(x, mode=mode).long()
    sub = torch.arange(n, device=dev) if n < 5000 else torch.cat(
        [torch.arange(2048, device=dev), torch.arange(n - 2048, n, device=dev)])
    want, near = _expected(dev, x[sub], mode)
    bad = (got[sub] != want) & ~near
    assert near.float().mean() < 0.02 and not bad.any(), sub[bad][:8].tolist()


def _integer_atoms(n, seed):
    rng = np.random.default_rng(seed)
    raw = cb.codebook_int8().astype(np.float32)
    a, b = rng.integers(1, 196561, n), rng.integers(1, 196561, n)
    sparse = np.zeros((n, 24), np.float32)
    for i in range(n):
        k = rng.integers(1, 25)
        sparse[i, rng.permutation(24)[:k]] = rng.choice([-2.0, 2.0], k)
    return torch.from_numpy(np.concatenate([
        raw[a] + raw[b], rng.integers(-4, 5, (n, 24)).astype(np.float32), 2 * raw[a], sparse]))


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("n", [700, 40_000])
def test_exact_ties(dev, mode, n):
    x = _integer_atoms(n, 5).to(dev)
    sub = torch.arange(0, len(x), max(1, len(x) // 2800), device=dev)
    got = castor.quantize_indices(x, mode=mode).long()[sub]
    want, _ = _expected(dev, x[sub], mode)
    assert torch.equal(got, want), int((got != want).sum())


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("n", [64, 98_304, 140_000])
def test_waves_full_of_tied_codes(dev, mode, n):
    # the atoms with the most tied words or octads among sparse integer vectors, repeated so that every wave's
    # survivor lists overflow (their rows then come from the sweeps after the first)
    pool = _integer_atoms(400, 9)[1200:].to(dev)
    a, c = _operands(dev, pool, mode)
    s = a @ c[1:].T
    ties = (s == s.max(1, keepdim=True).values).sum(1)
    top = pool[ties.argsort(descending=True)[:24]]
    assert int(ties.max()) > 40
    x = top.repeat((n + 23) // 24, 1)[:n].contiguous()
    got = castor.quantize_indices(x, mode=mode).long()
    want, _ = _expected(dev, top, mode)
    assert torch.equal(got, want.repeat((n + 23) // 24)[:n])


@pytest.mark.parametrize("mode", MODES)
def test_spiky_atoms(dev, mode):
    g = torch.Generator().manual_seed(11)
    x = torch.randn(4000, 24, generator=g) * 0.05
    x[torch.arange(4000), torch.randint(0, 24, (4000,), generator=g)] = torch.rand(4000, generator=g) * 8 + 1
    x = x.to(dev)
    got = castor.quantize_indices(x, mode=mode).long()
    want, near = _expected(dev, x, mode)
    bad = (got != want) & ~near
    assert not bad.any(), bad.nonzero()[:8].tolist()


@pytest.mark.parametrize("scale", [1e-7, 1e-3, 1e12, 2.0 ** 95, 1e36])
def test_pack_search_at_scale_limits(dev, scale):
    # fp32 scores would overflow from 2^96 on: those atoms are scanned code by code
    x = _atoms(300, 3, dev) * scale
    got = castor.quantize_indices(x, mode="pack").long()
    want, near = _expected(dev, x, "pack")
    bad = (got != want) & ~near
    assert not bad.any(), bad.nonzero()[:8].tolist()


@pytest.mark.parametrize("mode", MODES)
def test_non_finite_atoms_leave_the_others_alone(dev, mode):
    x = _atoms(3000, 4, dev)
    ref = castor.quantize_indices(x, mode=mode)
    bad = torch.arange(0, 3000, 97, device=dev)
    x[bad[0::2], 5] = float("nan")
    x[bad[1::2], 7] = float("-inf")
    got = castor.quantize_indices(x, mode=mode)
    keep = torch.ones(3000, dtype=torch.bool, device=dev)
    keep[bad] = False
    assert torch.equal(got[keep], ref[keep]) and int(got.min()) >= 0 and int(got.max()) <= 196560
    assert torch.all(got[bad[0::2]] == 0)  # a NaN coordinate: the origin
    if mode == "fp32":
        assert torch.all(got[bad] == 0)
