"""The error against 64 bits of launches that run whole (several waves of one
workgroup per item, no partitions): no larger than that of the launches in
partitions, or with other wave counts, that they replaced.  Each bound is the
relative norm measured for those on the same inputs."""
import pytest
import torch

import nanoinfer_amd as na

pytestmark = pytest.mark.gpu
L, H, D = 12, 12, 64
C = H * D


def _inputs(keys, nq, seqs, q8):
    """K and V that the cache holds exactly, and the queries of each sequence's last nq rows."""
    g = torch.Generator(device="cuda").manual_seed(keys + nq)
    out = []
    for _ in range(seqs):
        if q8:  # a row's largest value 127 steps of 2^-6: the scale is exact
            k, v = (torch.randint(-127, 128, (L, keys, H, D), device="cuda", generator=g).float() for _ in range(2))
            k[..., 0] = v[..., 0] = 127
            k, v = (x.reshape(L, keys, C) * 2.0 ** -6 for x in (k, v))
        else:
            k, v = (torch.randn((L, keys, C), device="cuda", generator=g).half().float() for _ in range(2))
        out.append((k, v, torch.randn((L, nq, C), device="cuda", generator=g)))
    return out


def _exact(q, k, v):
    nq, n = q.shape[1], k.shape[1]
    qh, kh, vh = (x.double().reshape(L, -1, H, D).transpose(1, 2).reshape(L * H, -1, D).contiguous() for x in (q, k, v))
    s = torch.matmul(qh, kh.transpose(1, 2).contiguous()) / D ** 0.5
    i, j = torch.arange(nq, device="cuda"), torch.arange(n, device="cuda")
    s.masked_fill_(j[None, :] > n - nq + i[:, None], -torch.inf)
    o = torch.matmul(torch.softmax(s, -1), vh)
    return o.reshape(L, H, nq, D).transpose(1, 2).reshape(L, nq, C)


@pytest.mark.parametrize("seqs,nq,keys,q8,bound", [
    (1, 1, 150, False, 1.40e-7), (1, 1, 517, False, 1.51e-7), (1, 1, 901, False, 1.64e-7), (1, 1, 1270, False, 1.77e-7),
    (1, 1, 3000, False, 1.84e-7), (3, 1, 900, False, 1.62e-7), (3, 1, 1270, False, 1.78e-7),
    (1, 1, 517, True, 0.94e-7), (1, 1, 901, True, 0.91e-7), (3, 1, 1270, True, 0.76e-7), (3, 1, 1500, True, 0.78e-7),
    (3, 1, 2000, False, 1.79e-7),  (1, 1, 3500, True, 0.75e-7),
    (1, 5, 300, False, 2.57e-7), (1, 5, 900, False, 2.65e-7), (1, 16, 900, False, 2.66e-7),
    (6, 5, 900, False, 2.92e-7), (13, 5, 700, False, 2.84e-7), (1, 5, 900, True, 0.93e-7), (6, 5, 900, True, 1.07e-7)])
def test_error_of_whole_launches(gpu, seqs, nq, keys, q8, bound):
    kv = na.PagedKv(na.BatchOpts(n_layer=L, n_head=H, head_dim=D, kv_blocks=seqs * (keys // 16 + 1), max_seqs=seqs,
                                 n_ctx=keys, max_rows=keys, q8=q8))
    data = _inputs(keys, nq, seqs, q8)
    rows = []
    for k, v, _ in data:
        s = kv.add_seq()
        kv.reserve(s, keys)
        kv.append([(s, i) for i in range(keys)], k, v)
        kv.commit(s, keys)
        rows += [(s, i) for i in range(keys - nq, keys)]
    got = kv.attention(torch.cat([q for _, _, q in data], 1), rows).double()
    want = torch.cat([_exact(q, k, v) for k, v, q in data], 1)
    err = float((got - want).norm() / want.norm())
    assert err <= bound, err
    kv.close()
