"""Contiguous attention of many queries (the matrix-core tile kernel) and its
edges: query blocks and key tiles of 16 with remainders, both head sizes and
both workgroup sizes, strided rows, and keys hidden from some queries that
hold infinities or NaN.

Bound against 64 bits, first order and worst case: a score is a sum of D
products, each |q_i k_i| / sqrt(D) off by at most D eps of itself (the q
scaling and the exponential's argument add 3 eps of the score), a weight is
off by as much in relative terms, and a sum over n keys by n eps more, in the
numerator and the denominator alike."""
import math

import numpy as np
import pytest
import torch

import nanoinfer_amd as na

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


def exact(q, k, v, p0, h, d):
    """The result and its error bound, in float64 on the CPU."""
    nq, n = q.shape[0], k.shape[0]
    out = np.empty((nq, h * d))
    bound = np.empty((nq, h * d))
    for i in range(h):
        s_ = slice(i * d, (i + 1) * d)
        qi, ki, vi = (x[:, s_].astype(np.float64) for x in (q, k, v))
        s = qi @ ki.T / math.sqrt(d)
        a = np.abs(qi) @ np.abs(ki).T / math.sqrt(d)
        hidden = np.arange(n)[None, :] > p0 + np.arange(nq)[:, None]
        s[hidden] = -np.inf
        a[hidden] = 0
        p = np.exp(s - s.max(1, keepdims=True))
        p /= p.sum(1, keepdims=True)
        out[:, s_] = p @ vi
        bound[:, s_] = (2 * ((d + 3) * EPS * a.max(1) + (n + 4) * EPS) * np.abs(vi).max())[:, None]
    return out, bound


@pytest.mark.parametrize("h,d,nq,p0", [
    (12, 64, 256, 0), (12, 64, 241, 15), (12, 64, 255, 1), (16, 64, 300, 16), (25, 64, 330, 7), (32, 128, 96, 0),
    (32, 128, 113, 31), (32, 128, 81, 50)])
def test_tile_kernel(gpu, h, d, nq, p0):
    g = torch.Generator(device="cuda").manual_seed(nq + p0)
    c = h * d
    n = p0 + nq
    qkv = torch.randn((n, 3 * c + 8), device="cuda", generator=g)
    q, k, v = qkv[p0:, :c], qkv[:, c:2 * c], qkv[:, 2 * c:3 * c]
    out = torch.full((nq, c + 4), 7.0, device="cuda")
    na.attention(q, k, v, nq, p0, h, d, out=out)
    got = out.cpu().numpy()
    assert (got[:, c:] == 7.0).all(), "wrote past the output rows' C columns"
    want, bound = exact(q.cpu().numpy(), k.cpu().numpy(), v.cpu().numpy(), p0, h, d)
    err = np.abs(got[:, :c] - want)
    assert (err <= bound).all(), f"max err {err.max():.2e}, bound {bound.min():.2e}"
    # f32 throughout: 1.0 to 1.4e-7 measured; an operand or the weights in 16 bits leave 1e-4 and more
    rel = np.linalg.norm(err) / np.linalg.norm(want)
    assert rel < 2e-7, rel
    # contiguous rows give the same bits as strided ones
    same = na.attention(q.contiguous(), k.contiguous(), v.contiguous(), nq, p0, h, d)
    assert torch.equal(same, out[:, :c])


@pytest.mark.parametrize("h,d,nq,p0", [(12, 64, 256, 0), (32, 128, 100, 5)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_hidden_keys_reach_no_query(gpu, h, d, nq, p0, bad):
    """A non-finite K or V row reaches the queries that see it and no other."""
    g = torch.Generator(device="cuda").manual_seed(5)
    c = h * d
    q = torch.randn((nq, c), device="cuda", generator=g)
    k, v = (torch.randn((p0 + nq, c), device="cuda", generator=g) for _ in range(2))
    at = p0 + 70  # query 70's own key
    want, bound = exact(*(x.cpu().numpy() for x in (q, k, v)), p0, h, d)
    for which in "kv":
        kk, vv = k.clone(), v.clone()
        (kk if which == "k" else vv)[at] = bad
        got = na.attention(q, kk, vv, nq, p0, h, d).cpu().numpy()
        err = np.abs(got[:70] - want[:70])
        assert (err <= bound[:70]).all(), which
        assert not np.isfinite(got[70:] if which == "v" or bad != bad else got[70:].sum(1)).any(), which


@pytest.mark.parametrize("h,d,nq,p0", [(12, 64, 21, 200), (12, 64, 22, 200), (32, 128, 8, 300), (32, 128, 9, 300)])
def test_row_kernel_wave_counts(gpu, h, d, nq, p0):
    """Few rows: 8 waves up to a row per CU, 4 beyond."""
    g = torch.Generator(device="cuda").manual_seed(6)
    c = h * d
    q = torch.randn((nq, c), device="cuda", generator=g)
    k, v = (torch.randn((p0 + nq, c), device="cuda", generator=g) for _ in range(2))
    want, bound = exact(*(x.cpu().numpy() for x in (q, k, v)), p0, h, d)
    got = na.attention(q, k, v, nq, p0, h, d).cpu().numpy()
    assert (np.abs(got - want) <= bound).all()


@pytest.mark.parametrize("h,d,nq,p0", [(12, 64, 256, 0), (12, 64, 640, 0), (32, 128, 100, 5)])
def test_large_values_stay_finite(gpu, h, d, nq, p0):
    """A later key's score 7.5 (base 2) above the first 16 keys': weights
    relative to those would be 181, times 60 keys or more of V up to 2e35 past
    f32's 3.4e38, though the result is their mean."""
    g = torch.Generator(device="cuda").manual_seed(7)
    c, n = h * d, p0 + nq
    a = math.sqrt(7.5 * math.log(2) / math.sqrt(d))
    q, k = (torch.full((r, c), a, device="cuda") for r in (nq, n))
    k[:16] = 0
    v = (1 + torch.rand((n, c), device="cuda", generator=g)) * 1e35
    want, bound = exact(*(x.cpu().numpy() for x in (q, k, v)), p0, h, d)
    got = na.attention(q, k, v, nq, p0, h, d).cpu().numpy()
    assert np.isfinite(got).all()
    assert (np.abs(got - want) <= bound).all()
