"""Launches with few (item, layer, head) units at head_dim 64 run one
workgroup per unit, no partitions and no merge launch, with a wave count that
depends on the units and the keys: both sides of each line (units per CU, keys
per item), f16 and Q8 caches, single rows and groups, a prompt chunk whose new
rows the attention launch appends, and rows of sequences without queries."""
import numpy as np
import pytest
import torch

import oracle
import nanoinfer_amd as na
from paged_mirror import Mirror, assert_close, mirror_step, step_rows

pytestmark = pytest.mark.gpu


def _opts(n_layer, n_head, q8, n_seqs, n_ctx):
    return na.BatchOpts(n_layer=n_layer, n_head=n_head, head_dim=64, q8=q8, kv_blocks=n_seqs * (n_ctx // 16 + 1),
                        max_seqs=n_seqs, n_ctx=n_ctx, max_rows=1024)


# contexts after the step, on both sides of 128 (4 waves), 384 and (Q8) 640 (16 waves), tile remainders among them
ROWS = [[1], [128], [129], [384], [385], [641], [1279], [1281], [2, 700, 17], [300] * 5, [30, 1000] + [90] * 19]


@pytest.mark.parametrize("per_layer", [False, True], ids=["all_layers", "per_layer"])
@pytest.mark.parametrize("ctx", ROWS, ids=lambda c: f"{len(c)}x{max(c)}")
def test_single_rows(gpu, oracle_lib, ctx, per_layer):
    rng = np.random.default_rng(len(ctx) + max(ctx))
    m = Mirror(_opts(2, 12, False, len(ctx) + 1, 1344))
    seqs = [m.kv.add_seq() for _ in ctx]
    for s, n in zip(seqs, ctx):
        m.fill(s, n - 1, rng)
    extra = m.kv.add_seq()
    for rnd in range(2):  # the second step appends one row further, and a mid-prompt chunk without a query
        work = [(s, 1, 1) for s in seqs] + ([(extra, 20, 0)] if rnd else [])
        rows, _ = step_rows(m.kv, work)
        q, k, v = (rng.standard_normal((2, len(rows), m.c)).astype(np.float32) for _ in range(3))
        m.kv.profile([2])
        got, want, qr = mirror_step(m, work, q, k, v, per_layer=per_layer)
        _, n_merge = m.kv.profile_read(2)
        m.kv.profile([])
        assert_close(got[:, qr], want[:, qr], f"round {rnd}")
        (kg, vg), (kw, vw) = m.gather(rows)
        assert np.array_equal(kg, kw) and np.array_equal(vg, vw)
        if max(ctx) + rnd <= 1280:
            assert n_merge == 0
    m.kv.close()


@pytest.mark.parametrize("per_layer", [False, True], ids=["all_layers", "per_layer"])
@pytest.mark.parametrize("ctx", [[128], [129], [640], [641], [1000, 3], [200] * 11], ids=lambda c: f"{len(c)}x{max(c)}")
def test_single_rows_q8(gpu, ctx, per_layer):
    """Against attention in float64 over the values the cache stores."""
    rng = np.random.default_rng(len(ctx) + max(ctx))
    L, H, D = 2, 12, 64
    kv = na.PagedKv(_opts(L, H, True, len(ctx), 1344))
    g = torch.Generator(device="cuda").manual_seed(1)
    seqs = [kv.add_seq() for _ in ctx]
    for s, n in zip(seqs, ctx):
        if n > 1:
            k, v = (torch.randn((L, n - 1, H * D), device="cuda", generator=g) for _ in range(2))
            kv.reserve(s, n - 1)
            for p in range(0, n - 1, 512):
                e = min(n - 1, p + 512)
                kv.append([(s, i) for i in range(p, e)], k[:, p:e], v[:, p:e])
            kv.commit(s, n - 1)
    q, k, v = (torch.randn((L, len(ctx), H * D), device="cuda", generator=g) for _ in range(3))
    work = [(s, 1, 1) for s in seqs]
    if per_layer:
        out = torch.zeros_like(q)
        kv.step_begin(work)
        for l in range(L):
            kv.step_layer(l, q[l], k[l], v[l], out=out[l])
        kv.step_end()
    else:
        out = kv.step(work, q, k, v)
    for i, (s, n) in enumerate(zip(seqs, ctx)):
        parts = [kv.gather_q8([(s, j) for j in range(p, min(n, p + 512))]) for p in range(0, n, 512)]
        (kq, vq), (ks, vs) = ([torch.cat([x[a][b] for x in parts], 1) for b in range(2)] for a in range(2))
        kf, vf = ((x.double().reshape(L, n, H, D) * sc.double()[..., None]).cpu().numpy() for x, sc in ((kq, ks), (vq, vs)))
        # the new row is stored as the standalone quantiser would store it
        x = k[:, i].reshape(L, H, D).cpu().numpy()
        scale = (np.abs(x).max(-1) / np.float32(127)).astype(np.float32)
        assert np.array_equal(ks[:, -1].cpu().numpy(), scale)
        qi = q[:, i].reshape(L, H, D).double().cpu().numpy()
        sc = np.einsum("lhd,lnhd->lhn", qi, kf) / 8
        p = np.exp(sc - sc.max(-1, keepdims=True))
        want = np.einsum("lhn,lnhd->lhd", p / p.sum(-1, keepdims=True), vf).reshape(L, H * D)
        assert_close(out[:, i].cpu().numpy(), want, f"sequence {i} ({n} keys)")
    kv.close()


@pytest.mark.parametrize("n_seqs,nq,ctx", [(1, 2, 40), (2, 16, 300), (9, 5, 1230), (21, 5, 333), (22, 5, 333)])
def test_groups(gpu, oracle_lib, n_seqs, nq, ctx):
    """Verify groups below, at and past two workgroups per CU (21 and 22
    sequences x 2 layers x 12 heads: 504 and 528 units), and one queried row
    after a long chunk of new rows."""
    rng = np.random.default_rng(n_seqs * 100 + nq)
    m = Mirror(_opts(2, 12, False, n_seqs, 1344))
    seqs = [m.kv.add_seq() for _ in range(n_seqs)]
    for i, s in enumerate(seqs):
        m.fill(s, max(1, ctx - 13 * i), rng)
    for work in ([(s, nq, nq) for s in seqs], [(seqs[0], 45, 1)]):
        for per_layer in (False, True):
            rows, _ = step_rows(m.kv, work)
            q, k, v = (rng.standard_normal((2, len(rows), m.c)).astype(np.float32) for _ in range(3))
            m.kv.profile([2])
            base = [m.kv.seq_len(s) for s in seqs]
            got, want, qr = mirror_step(m, work, q, k, v, per_layer=per_layer)
            _, n_merge = m.kv.profile_read(2)
            m.kv.profile([])
            assert n_merge == 0
            assert_close(got[:, qr], want[:, qr], f"{work[0]} per_layer {per_layer}")
            (kg, vg), (kw, vw) = m.gather(rows)
            assert np.array_equal(kg, kw) and np.array_equal(vg, vw)
            for s, n in zip(seqs, base):
                m.kv.truncate(s, n)
    m.kv.close()


@pytest.mark.parametrize("q8", [False, True], ids=["f16", "q8"])
@pytest.mark.parametrize("n_layer,nq,ctx,whole", [
    (1, 1, [4090] + [100] * 7, False), (1, 1, [4090] + [100] * 31, False), (12, 1, [4090, 100], False),
    (1, 1, [2000] * 16, True), (12, 1, [1500], True), (1, 1, [1280] + [100] * 7, True), (12, 1, [1280] * 2, True),
    (1, 5, [2000] + [100] * 7, False), (2, 16, [1280], False), (1, 5, [4090] + [100] * 7, False),
    (1, 5, [2000] * 16, True), (12, 5, [1500], True), (1, 16, [1280] + [100] * 7, True)],
    ids=lambda x: f"{len(x)}x{x[0]}" if isinstance(x, list) else str(x))
def test_long_items_run_whole_beside_enough_others(gpu, n_layer, nq, ctx, whole, q8):
    """A launch waits for its longest whole item: one long context among short
    ones goes in partitions (and a merge launch), as many as it fills the GPU
    with stay whole.  The results agree with partitions of 256 keys (f32 sums
    or f16 pairs in another order: 4e-6 of the norm)."""
    kv = na.PagedKv(na.BatchOpts(n_layer=n_layer, n_head=12, head_dim=64, q8=q8, kv_blocks=sum(c // 16 + 1 for c in ctx),
                                 max_seqs=len(ctx), n_ctx=max(ctx), max_rows=2048))
    g = torch.Generator(device="cuda").manual_seed(3)
    rows = []
    for c in ctx:
        s = kv.add_seq()
        kv.reserve(s, c)
        for p in range(0, c, 2048):
            n = min(c, p + 2048) - p
            k, v = (torch.randn((n_layer, n, 768), device="cuda", generator=g) for _ in range(2))
            kv.append([(s, p + i) for i in range(n)], k, v)
        kv.commit(s, c)
        rows += [(s, c - nq + i) for i in range(nq)]
    q = torch.randn((n_layer, len(rows), 768), device="cuda", generator=g)
    kv.profile([2])
    got = kv.attention(q, rows)
    torch.cuda.synchronize()
    _, n_merge = kv.profile_read(2)
    kv.profile([])
    assert n_merge == (0 if whole else 1)
    want = kv.attention(q, rows, split_tokens=256).double()
    assert (got - want).norm() / want.norm() < 4e-6
    kv.close()
