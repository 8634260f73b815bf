"""plx_prefill_attention at the edges of its 64-query, 64-key tiles, against float64.

The bar per element, 64 * 2^-24 * max|V| (and 1e-5 relative over all), covers fp32 scores of 24-term dot
products of rows of norm sqrt 24 (|score| <= sqrt 24 here, so a rounding of it moves a probability by
sqrt 24 * 24 * 2^-24 relative) and the fp32 sums of probabilities and values.
"""

import math

import pytest
import torch

from pollux_amd.model import RMSNorm, prefill_attention

pytestmark = pytest.mark.gpu


def _norm(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-8) * w


def _case(dev, b, heads, t, p0, max_len, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    q, k, v = (torch.randn(b, t, heads * 24, generator=g, device=dev) for _ in range(3))
    kc, vc = (torch.randn(b, heads, max_len, 24, generator=g, device=dev) for _ in range(2))
    q_ln, k_ln = RMSNorm(24).to(dev), RMSNorm(24).to(dev)
    with torch.no_grad():
        q_ln.weight.copy_(1 + 0.1 * torch.randn(24, generator=g, device=dev))
        k_ln.weight.copy_(1 + 0.1 * torch.randn(24, generator=g, device=dev))
    return q, k, v, kc, vc, q_ln, k_ln


def _heads(x, heads):
    return x.view(*x.shape[:2], heads, 24).transpose(1, 2).double().contiguous()


@pytest.mark.parametrize("b,heads,t,p0,max_len", [
    (1, 3, 63, 0, 63), (1, 3, 64, 0, 80), (2, 3, 65, 0, 65), (1, 2, 16, 0, 16), (1, 2, 17, 63, 90), (1, 2, 2, 64, 70),
    (1, 2, 100, 65, 200), (3, 1, 129, 1, 130), (1, 5, 1024, 0, 1024), (2, 2, 191, 127, 400), (2, 40_000, 1, 0, 1)])
def test_tile_edges(dev, b, heads, t, p0, max_len):
    q, k, v, kc, vc, q_ln, k_ln = _case(dev, b, heads, t, p0, max_len, t + p0)
    kc0, vc0 = kc.clone(), vc.clone()
    with torch.no_grad():
        out = prefill_attention(q, k, v, q_ln, k_ln, kc, vc, p0)
        qn, kn, vn = _norm(_heads(q, heads), q_ln.weight.double()), _norm(_heads(k, heads), k_ln.weight.double()), _heads(v, heads)
        keys = torch.cat([kc0[:, :, :p0].double(), kn], 2)
        vals = torch.cat([vc0[:, :, :p0].double(), vn], 2)
        s = qn @ keys.transpose(-1, -2).contiguous() / math.sqrt(24)
        s = s.masked_fill(~torch.ones(t, p0 + t, dtype=torch.bool, device=dev).tril(p0), -math.inf)
        ref = (torch.softmax(s, -1) @ vals).transpose(1, 2).reshape(b, t, heads * 24)
    err = (out.double() - ref).abs().max().item()
    rel = ((out.double() - ref).norm() / ref.norm()).item()
    print(f"[prefill] b={b} H={heads} t={t} p0={p0}: max {err:.2e} rel {rel:.2e}", flush=True)
    assert err <= 64 * 2.0 ** -24 * vals.abs().max().item() and rel <= 1e-5
    new = slice(p0, p0 + t)
    assert ((kc[:, :, new].double() - kn).abs() <= 2e-6 * kn.abs() + 1e-30).all()
    assert torch.equal(vc[:, :, new], _heads(v, heads).float())
    kc[:, :, new], vc[:, :, new] = kc0[:, :, new], vc0[:, :, new]
    assert torch.equal(kc, kc0) and torch.equal(vc, vc0)


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("row", [0, 5, 40, 70, 127])
def test_a_bad_row_reaches_no_earlier_query(dev, bad, row):
    q, k, v, kc, vc, q_ln, k_ln = _case(dev, 2, 2, 130, 10, 140, 5)
    with torch.no_grad():
        ref = prefill_attention(q, k, v, q_ln, k_ln, kc.clone(), vc.clone(), 10)
        v[1, row, 3] = bad
        k[1, row, 30] = bad
        out = prefill_attention(q, k, v, q_ln, k_ln, kc, vc, 10)
    assert torch.equal(out[0], ref[0])
    tol = 64 * 2.0 ** -24 * ref.abs().max().item()
    assert ((out[1, :row] - ref[1, :row]).abs() <= tol).all()
    assert not torch.isfinite(out[1, row:, 3]).any() and torch.isnan(out[1, row:, 24:]).all()


@pytest.mark.parametrize("size", [30.0, 1e3, 1e5, 1e9])
def test_scores_of_any_size(dev, size):
    # norm weights far from 1 (scores up to 24 size^2): where one key's score leads by more than the fp32 roundings of
    # the two (24 * 2^-24 of the products' sizes each) and the softmax's own width, the output is its value
    b, heads, t, p0 = 1, 3, 200, 70
    q, k, v, kc, vc, q_ln, k_ln = _case(dev, b, heads, t, p0, 300, 8)
    with torch.no_grad():
        q_ln.weight.mul_(size)
        k_ln.weight.mul_(size)
        kc.mul_(size)
        out = prefill_attention(q, k, v, q_ln, k_ln, kc.clone(), vc.clone(), p0)
        qn, kn = _norm(_heads(q, heads), q_ln.weight.double()), _norm(_heads(k, heads), k_ln.weight.double())
        keys = torch.cat([kc[:, :, :p0].double(), kn], 2)
        vals = torch.cat([vc[:, :, :p0].double(), _heads(v, heads)], 2)
        mask = ~torch.ones(t, p0 + t, dtype=torch.bool, device=dev).tril(p0)
        s = (qn @ keys.transpose(-1, -2).contiguous() / math.sqrt(24)).masked_fill(mask, -math.inf)
        unsure = 24 * 2.0 ** -24 * (qn.abs() @ keys.abs().transpose(-1, -2).contiguous()).max(-1).values / math.sqrt(24)
        top = s.topk(2, -1)
        lead = top.values[..., 0] - top.values[..., 1] > 2 * unsure + 30
        want = vals.gather(2, top.indices[..., :1].expand(-1, -1, -1, 24))
    got = _heads(out, heads)
    assert torch.isfinite(out).all() and lead.float().mean() > 0.3
    assert ((got - want)[lead].abs() <= 1e-6 * vals.abs().max()).all()
