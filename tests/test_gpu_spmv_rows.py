"""BSR matrix-vector product over rows of any length: shorter and longer than
the blocks a row keeps in flight, empty rows, row counts that do not fill the
last wavefront."""
import numpy as np
import pytest

import gpu_fem_amd as G
from gpu_helpers import dev, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,longest", [(1, 1), (9, 3), (10, 9), (11, 10),
                                       (41, 18), (200, 19), (333, 60)])
def test_row_lengths(gpu_ctx, n, longest, dtype):
    import torch

    print(f"[gpu] spmv n={n} rows up to {longest}", flush=True)
    rng = np.random.default_rng(n)
    longest = min(longest, n)
    length = rng.integers(0, longest + 1, n)
    length[0] = longest
    rowp = np.concatenate([[0], np.cumsum(length)]).astype(np.int32)
    cols = np.concatenate([np.sort(rng.choice(n, k, replace=False))
                           for k in length]).astype(np.int32)
    a = rng.standard_normal((len(cols), 6, 6)).astype(dtype)
    x = rng.standard_normal(6 * n).astype(dtype)
    d_y = torch.full((6 * n,), np.nan, device="cuda",
                     dtype=torch.float64 if dtype == np.float64 else torch.float32)
    d_rp, d_c, d_a, d_x = dev(rowp), dev(cols), dev(a), dev(x)
    fn = (G.lib().gf_bsr_spmv_f64 if dtype == np.float64
          else G.lib().gf_bsr_spmv_f32)
    gpu_ctx.check(fn(gpu_ctx.h, n, G.ptr(d_rp), G.ptr(d_c), G.ptr(d_a),
                     G.ptr(d_x), G.ptr(d_y)))
    gpu_ctx.sync()
    y = host(d_y)
    rows = np.repeat(np.arange(n), length)
    xb = x.reshape(n, 6).astype(np.longdouble)[cols]
    ref, mag = np.zeros((n, 6), np.longdouble), np.zeros((n, 6), np.longdouble)
    ad = a.astype(np.longdouble)
    np.add.at(ref, rows, np.einsum("kij,kj->ki", ad, xb))
    np.add.at(mag, rows, np.einsum("kij,kj->ki", np.abs(ad), np.abs(xb)))
    # a sum of at most 6 * longest products, each term rounded once
    tol = (6 * longest + 1) * np.finfo(dtype).eps * mag.ravel()
    assert np.all(np.abs(y - ref.ravel()) <= tol)
