"""The QKV projection's feature tiles of large batches: 16, 32 and 48 features
wide by the row count.  Every output is summed in the same order whatever the
tile, so each width has the bits of a 17-row batch (another kernel, one tile
of rows) and is within f32 rounding of the product in 64 bits: |y - y64| <=
768 * 2^-24 * sum |x w| bounds any order, and sum |x w| of 768 products of
N(0,1) x N(0,1/768) stays below 40, so 2e-3; 8 parts of 96 random roundings each
leave ~1e-6, held here to 2e-5."""
import numpy as np
import pytest
import torch

import oracle
import nanoinfer_amd as na
from nanoinfer_amd import workloads

pytestmark = pytest.mark.gpu


# 12 x 64 on 256 CUs: 16-wide up to 384 rows, 32-wide at 385..448, 16-wide at 449, 48-wide at 512, 32-wide at 520
# (f32: 16-wide) and 640; 900 rows leave 4 rows in the last tile.
@pytest.mark.parametrize("n", [384, 385, 417, 448, 449, 512, 520, 640, 900])
@pytest.mark.parametrize("fmt", ["f32", "f16", "q8_0", "q4_0"])
def test_tile_widths_agree(gpu, oracle_lib, n, fmt):
    kv = na.PagedKv(na.BatchOpts(**workloads.GPT2, kv_blocks=8, max_seqs=2, n_ctx=64, max_rows=1024))
    c, d_in = kv.opts.n_embd, 784 if fmt in ("f32", "f16") else 800  # a last chunk that is not full
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, d_in)).astype(np.float32)
    w = (rng.standard_normal((3 * c, d_in)) / np.sqrt(d_in)).astype(np.float32)
    b = (rng.standard_normal(3 * c) * 0.1).astype(np.float32)
    wd = torch.from_numpy(w if fmt == "f32" else oracle.quantize(w, fmt)).cuda()
    if fmt != "f32":
        w = oracle.dequantize(wd.cpu().numpy(), w.size, fmt).reshape(w.shape)
    xd, bd = torch.from_numpy(x).cuda(), torch.from_numpy(b).cuda()
    got = kv.qkv_project(xd, wd, bd, w_format=fmt).cpu().numpy()
    assert np.abs(got - oracle.matvec_f64(x, w, b)).max() < 2e-5
    for r in (0, n - 17):
        few = kv.qkv_project(xd[r:r + 17], wd, bd, w_format=fmt).cpu().numpy()
        assert np.array_equal(few.view(np.uint32), got[r:r + 17].view(np.uint32)), (n, r)
