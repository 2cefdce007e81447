"""The Python calls take the same tensors whichever form they come in: plain
tensors (checked quickly), tensor subclasses, allocated or given outputs, row
and work lists as lists, arrays, strided or read-only arrays."""
import numpy as np
import pytest
import torch

import nanoinfer_amd as na

pytestmark = pytest.mark.gpu
L, H, D, N = 2, 2, 64, 5
C = H * D


def _forms(rows):
    a = np.array(rows, np.uint32)
    ro = a.copy()
    ro.flags.writeable = False
    return [rows, a, ro, np.repeat(a, 2, 0)[::2], a.astype(np.int64)]


def test_forms_agree(gpu):
    g = torch.Generator(device="cuda").manual_seed(2)
    kv = na.PagedKv(na.BatchOpts(n_layer=L, n_head=H, head_dim=D, kv_blocks=16, max_seqs=2, n_ctx=64, max_rows=16))
    s = kv.add_seq()
    q, k, v = (torch.randn((L, N, C), device="cuda", generator=g) for _ in range(3))
    x, w = torch.randn((N, C), device="cuda", generator=g), torch.randn((3 * C, C), device="cuda", generator=g)
    param = lambda t: torch.nn.Parameter(t, requires_grad=False)
    work, rows = [(s, N, N)], [(s, i) for i in range(N)]
    want = kv.step(work, q, k, v)
    for wk in _forms(work):
        for wrap in (lambda t: t, param):
            kv.truncate(s, 0)
            out = torch.zeros_like(q)
            assert kv.step(wk, wrap(q), wrap(k), wrap(v), out=out) is out
            assert torch.equal(out, want)
            kv.truncate(s, 0)
            kv.step_begin(wk)
            got = [kv.step_layer(l, wrap(q[l]), wrap(k[l]), wrap(v[l])) for l in range(L)]
            kv.step_end()
            for l in range(L):
                torch.testing.assert_close(got[l], want[l], rtol=1e-5, atol=1e-5)
    want_a = kv.attention(q, rows)
    want_l = kv.attention(q[1], rows, layer=1)
    want_q = kv.qkv_append(rows, x, w, layer=0)
    for r in _forms(rows):
        out = torch.zeros_like(q)
        assert torch.equal(kv.attention(param(q), r, out=out)[1], want_a[1])
        assert torch.equal(kv.attention(q[1], r, layer=1, out=out[0]), want_l)
        assert torch.equal(kv.qkv_append(r, x, w, layer=0, q_out=out[0]), want_q)
        assert torch.equal(kv.qkv_append(r, param(x), param(w), layer=0), want_q)
    rows_out = na.attention(x, x, x, N, 0, H, D)
    out = torch.zeros((N, C + 4), device="cuda")
    assert torch.equal(na.attention(param(x), x, x, N, 0, H, D, out=out[:, :C]), rows_out)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # the current stream, and a stream given by the caller
        a = na.attention(x, x, x, N, 0, H, D, out=torch.zeros_like(x))
    b = na.attention(x, x, x, N, 0, H, D, out=out[:, :C], stream=side)
    side.synchronize()
    assert torch.equal(a, rows_out) and torch.equal(b, rows_out)
    for bad in (q.cpu(), q[:, :3], q.double()):
        with pytest.raises((TypeError, ValueError)):
            kv.attention(bad, rows)
        with pytest.raises((TypeError, ValueError)):
            kv.attention(q, rows, out=bad)
    with pytest.raises((TypeError, ValueError)):
        kv.qkv_append(rows, x, w.cpu(), layer=0, q_out=torch.zeros_like(x))
    kv.close()
