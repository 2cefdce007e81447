"""Launches of prompt chunks run as 64-row prefill groups or as 16-row groups
on the group kernel, whichever the launch's size makes faster, in one launch
either way (a run's short last group joins the others').  Both sides of the
rule against the oracle, and against the same rows planned as prefill groups
(an explicit partition size keeps those)."""
import numpy as np
import pytest
import torch

import oracle
import nanoinfer_amd as na
from paged_mirror import Mirror, assert_close, mirror_step, step_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("per_layer", [False, True], ids=["all_layers", "per_layer"])
@pytest.mark.parametrize("ctx,rows", [([0], [17]), ([0], [65]), ([0, 3], [80, 64]), ([300], [33]), ([0], [200]),
                                      ([100, 0, 7], [200, 129, 18])], ids=str)
def test_prompt_steps(gpu, oracle_lib, head_dim, per_layer, ctx, rows):
    rng = np.random.default_rng(sum(rows) + sum(ctx))
    opts = na.BatchOpts(n_layer=2, n_head=768 // head_dim, head_dim=head_dim, kv_blocks=120, max_seqs=len(ctx),
                        n_ctx=512, max_rows=1024)
    m = Mirror(opts)
    seqs = [m.kv.add_seq() for _ in ctx]
    for s, n in zip(seqs, ctx):
        if n:
            m.fill(s, n, rng)
    work = [(s, n, n) for s, n in zip(seqs, rows)]
    r, _ = step_rows(m.kv, work)
    q, k, v = (rng.standard_normal((2, len(r), m.c)).astype(np.float32) for _ in range(3))
    m.kv.profile([1])
    got, want, qr = mirror_step(m, work, q, k, v, per_layer=per_layer)
    _, n_attn = m.kv.profile_read(1)
    m.kv.profile([])
    assert n_attn == (2 if per_layer else 1)
    assert_close(got[:, qr], want[:, qr], "step")
    (kg, vg), (kw, vw) = m.gather(r)
    assert np.array_equal(kg, kw) and np.array_equal(vg, vw)
    m.kv.close()


@pytest.mark.parametrize("q8", [False, True], ids=["f16", "q8"])
@pytest.mark.parametrize("n_layer,ctx,rows", [(1, 0, 64), (1, 0, 80), (1, 300, 20), (1, 0, 509), (2, 250, 100),
                                              (12, 0, 64), (12, 0, 80), (12, 300, 20), (12, 300, 100), (1, 1500, 40)])
def test_same_rows_as_prefill_groups(gpu, q8, n_layer, ctx, rows):
    """Strided q and out, one sequence; two summation orders of f32 values
    carried as f16 pairs (2^-22 of each): 4e-6 of the result's norm."""
    n = ctx + rows
    kv = na.PagedKv(na.BatchOpts(n_layer=n_layer, n_head=12, head_dim=64, kv_blocks=n // 16 + 1, max_seqs=1,
                                 n_ctx=n, max_rows=n, q8=q8))
    g = torch.Generator(device="cuda").manual_seed(rows)
    s = kv.add_seq()
    kv.reserve(s, n)
    k, v = (torch.randn((n_layer, n, 768), device="cuda", generator=g) for _ in range(2))
    kv.append([(s, i) for i in range(n)], k, v)
    kv.commit(s, n)
    q = torch.randn((n_layer, rows + 3, 772), device="cuda", generator=g)[:, :rows, :768]
    at = [(s, ctx + i) for i in range(rows)]
    want = kv.attention(q, at, split_tokens=4096)
    out = torch.full((n_layer, rows, 1536), 7.0, device="cuda")
    kv.attention(q, at, out=out[:, :, :768])
    assert (out[:, :, 768:] == 7.0).all()
    err = (out[:, :, :768] - want).double().norm() / want.double().norm()
    assert err < 4e-6, err
    one = kv.attention(q[0], at, layer=0)
    err = (one - want[0]).double().norm() / want[0].double().norm()
    assert err < 4e-6, err
    kv.close()
