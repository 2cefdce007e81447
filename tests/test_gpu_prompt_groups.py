"""Launches of prompt chunks run as 64-row prefill groups or as 16-row groups
on the group kernel, whichever the launch's size makes faster.  Both sides of
the rule against the oracle, and against the same rows planned as prefill
groups (an explicit partition size keeps those).  A run's last 1..16 rows past
a multiple of 64 stay out of the prefill launch: one row keeps f32 queries and
weights, more keep the group kernel's error, and split they keep its small
partials."""
import numpy as np
import pytest
import torch

import oracle
import nanoinfer_amd as na
from nanoinfer_amd import _abi
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
    tail = any(n > 64 and 0 < n % 64 <= 16 for n in rows)  # a launch of its own after prefill groups
    assert n_attn in ((2, 4) if tail and per_layer else (1, 2) if tail else (2,) if per_layer else (1,))
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


def _prompt(n_layer, ctx, rows, head_dim, g, c=768):
    """One sequence of ctx + rows positions, its K/V in the cache, and q for the last `rows`."""
    n, h = ctx + rows, c // head_dim
    kv = na.PagedKv(na.BatchOpts(n_layer=n_layer, n_head=h, head_dim=head_dim, kv_blocks=n // 16 + 1, max_seqs=1,
                                 n_ctx=n, max_rows=n))
    s = kv.add_seq()
    kv.reserve(s, n)
    k, v = (torch.randn((n_layer, n, c), device="cuda", generator=g).half().float() for _ in range(2))
    kv.append([(s, i) for i in range(n)], k, v)
    kv.commit(s, n)
    q = torch.randn((n_layer, rows, c), device="cuda", generator=g)
    return kv, [(s, ctx + i) for i in range(rows)], q, k, v


def _exact(q, k, v, ctx, head_dim):
    """Attention in float64 of q's rows at positions ctx.. over k, v [n, 768]."""
    nq, n, h = q.shape[0], k.shape[0], 768 // head_dim
    qh, kh, vh = (x.double().reshape(-1, h, head_dim).transpose(0, 1).contiguous() for x in (q, k, v))
    s = torch.matmul(qh, kh.transpose(1, 2).contiguous()) / head_dim ** 0.5
    i, j = torch.arange(nq, device="cuda"), torch.arange(n, device="cuda")
    s.masked_fill_(j[None, :] > ctx + i[:, None], -np.inf)
    return torch.matmul(torch.softmax(s, -1), vh).transpose(0, 1).reshape(nq, 768)


def _rel(got, want):
    return float((got.double() - want).norm() / want.norm())


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("n_layer,ctx,rows", [(12, 0, 65), (12, 0, 129), (12, 150, 193), (1, 0, 65), (1, 0, 513),
                                              (1, 300, 129)], ids=str)
def test_a_single_last_row_is_f32(gpu, n_layer, ctx, rows, head_dim):
    """The row a prompt's first token comes from.  Its query scaled past f16's
    range (2^19 |q| log2(e) / sqrt(head_dim): past 65504 an f16 pair is
    infinite) still finds its best key: the scores of two keys differ by far
    more than f32's rounding of them, so the result is that key's V."""
    g = torch.Generator(device="cuda").manual_seed(rows)
    kv, at, q, k, v = _prompt(n_layer, ctx, rows, head_dim, g)
    q[:, -1] *= 2.0 ** 19
    got = kv.attention(q, at)[:, -1:]
    for l in range(n_layer):
        assert _rel(got[l], _exact(q[l, -1:], k[l], v[l], ctx + rows - 1, head_dim)) < 1e-6, l
    kv.close()


@pytest.mark.parametrize("n_layer,ctx,rows", [(12, 0, 70), (12, 0, 200), (12, 150, 400)], ids=str)
def test_a_short_last_group_has_the_group_kernels_error(gpu, n_layer, ctx, rows):
    """Against the same rows attended on their own: the same kernel over the
    same keys, partitioned by the launch's size, 1.25 times apart at most."""
    g = torch.Generator(device="cuda").manual_seed(rows)
    kv, at, q, k, v = _prompt(n_layer, ctx, rows, 64, g)
    t = rows % 64
    both, alone = kv.attention(q, at)[:, -t:], kv.attention(q[:, -t:].contiguous(), at[-t:])
    want = torch.stack([_exact(q[l, -t:], k[l], v[l], ctx + rows - t, 64) for l in range(n_layer)])
    assert _rel(both, want) < 1.25 * _rel(alone, want)
    kv.close()


@pytest.mark.parametrize("rows", [65, 80])
def test_a_split_last_group_fits_the_noalloc_scratch(gpu, rows):
    """8 partitions x (64 rows, and a last group of 1 or 16) of 144 (layer,
    head)s stay below the 32 MiB of ni_kv_step_noalloc, and its results are
    ni_kv_step's."""
    g = torch.Generator(device="cuda").manual_seed(rows)
    ctx, n = 1024 - rows, 1024
    q, k, v = (torch.randn((12, n, 768), device="cuda", generator=g) for _ in range(3))
    work = np.array([[0, rows, rows]], np.uint32)
    outs = []
    for fn in (_abi.lib().ni_kv_step, _abi.lib().ni_kv_step_noalloc):
        kv = na.PagedKv(na.BatchOpts(n_layer=12, n_head=12, head_dim=64, kv_blocks=64, max_seqs=1, n_ctx=n, max_rows=n))
        s = kv.add_seq()
        kv.reserve(s, ctx)
        kv.append([(s, i) for i in range(ctx)], k[:, :ctx], v[:, :ctx])
        kv.commit(s, ctx)
        qn, kn, vn = (x[:, ctx:].contiguous() for x in (q, k, v))
        out = torch.full_like(qn, float("nan"))
        rc = fn(kv.handle, _abi.C.cast(work.ctypes.data, _abi.C.POINTER(_abi.ni_work)), 1, qn.data_ptr(), kn.data_ptr(),
                vn.data_ptr(), qn.stride(1), qn.stride(0), out.data_ptr(), out.stride(1), out.stride(0), 128,
                torch.cuda.current_stream().cuda_stream)
        assert rc == 0, _abi.lib().ni_kv_last_error(kv.handle).decode()
        torch.cuda.synchronize()
        outs.append(out)
        kv.close()
    assert torch.equal(*outs)


@pytest.mark.parametrize("n_layer,head_dim,ctx,rows,tiles", [
    (1, 64, 0, 509, True), (1, 64, 1300, 64, True), (12, 64, 0, 200, True), (12, 64, 700, 32, True),
    (12, 64, 0, 512, False), (12, 64, 5000, 64, False), (12, 64, 9000, 64, False), (1, 64, 0, 513, True),
    (1, 128, 0, 250, True), (1, 128, 1500, 64, True), (2, 128, 500, 64, False), (1, 128, 0, 500, False)], ids=str)
def test_which_groups_run(gpu, n_layer, head_dim, ctx, rows, tiles):
    """Prefill groups and tile groups of the same rows differ in rounding, so the
    bits of a launch with the automatic cut are a prefill launch's (an explicit
    partition size, as large as the automatic one) exactly where the rule says
    so: 16-row groups where they are faster with all their launches, the merge
    of their partitions and the row launch of a single last row included."""
    g = torch.Generator(device="cuda").manual_seed(rows)
    kv, at, q, _, _ = _prompt(n_layer, ctx, rows, head_dim, g, 768 if head_dim == 64 else 4096)
    same = torch.equal(kv.attention(q, at), kv.attention(q, at, split_tokens=4096))
    assert same != tiles
    kv.close()
