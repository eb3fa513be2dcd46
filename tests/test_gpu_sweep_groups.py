"""Triangular sweeps over row groups (trsv_group_kernel) against the oracle's
sweeps: groups of one to eight rows, records shared by several groups,
patterns that are not symmetric, rows of several passes, the smallest systems
and those on either side of the rule that chooses between groups and rows."""
import numpy as np
import pytest

import gpu_fem_amd as G
import oracle
from gpu_helpers import dev, host

pytestmark = pytest.mark.gpu


def pattern(n, kind, seed=0):
    """Sorted block pattern with a full diagonal."""
    import scipy.sparse as sp

    rng = np.random.default_rng(seed)
    if kind == "dense":
        m = sp.csr_matrix(np.ones((n, n)))
    elif kind == "chain":  # tridiagonal: groups of eight rows
        m = sp.diags([1.0, 1.0, 1.0], [-1, 0, 1], shape=(n, n))
    elif kind == "band":  # 40 blocks on either side: several passes
        m = sp.diags([1.0] * 81, range(-40, 41), shape=(n, n))
    elif kind == "forest":  # chains of 1 to 5 rows, interleaved
        rows, cols, i = [], [], 0
        perm = rng.permutation(n)
        while i < n:
            k = int(rng.integers(1, 6))
            c = np.sort(perm[i:i + k])
            rows += list(c[1:]) + list(c[:-1])
            cols += list(c[:-1]) + list(c[1:])
            i += k
        rows += list(range(n)) + [n - 1] * n + list(range(n))
        cols += list(range(n)) + list(range(n)) + [n - 1] * n
        m = sp.csr_matrix((np.ones(len(rows)), (rows, cols)), shape=(n, n))
    else:  # random, not symmetric
        m = sp.random(n, n, min(1.0, 6.0 / n), random_state=seed) + sp.eye(n)
        if kind == "lower":
            m = sp.tril(m)
        elif kind == "chained":
            m = m + sp.diags([1.0, 1.0], [-1, 1], shape=(n, n))
    m = sp.csr_matrix(m)
    m.sum_duplicates()
    m.sort_indices()
    return m.indptr.astype(np.int32), m.indices.astype(np.int32)


def factors(rowp, cols, seed):
    """Factor values whose sweeps are well conditioned: off-diagonal blocks of
    row sums below 1/2, diagonal entries of U in [1, 2]."""
    rng = np.random.default_rng(seed)
    n = len(rowp) - 1
    rows = np.repeat(np.arange(n), np.diff(rowp))
    v = rng.uniform(-1.0, 1.0, (len(cols), 6, 6)) / (
        12.0 * np.diff(rowp))[rows][:, None, None]
    d = np.nonzero(rows == cols)[0]
    for a in range(6):
        v[d, a, a] = rng.uniform(1.0, 2.0, n)
    return v.ravel()


CASES = [("dense", 1), ("dense", 2), ("dense", 9), ("dense", 30),
         ("chain", 7), ("chain", 8), ("chain", 65), ("chain", 1000),
         ("band", 333), ("forest", 64), ("forest", 1500), ("random", 400),
         ("lower", 300), ("chained", 500)]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind,n", CASES)
def test_sweeps_match_oracle(gpu_ctx, kind, n, dtype):
    import torch

    print(f"[gpu] group sweeps {kind} n={n} {np.dtype(dtype).name}", flush=True)
    rowp, cols = pattern(n, kind, seed=n)
    lu = factors(rowp, cols, n + 1).astype(dtype)
    b = np.random.default_rng(n + 2).standard_normal(6 * n).astype(dtype)
    x_o = oracle.bsr_trsv(rowp, cols, lu.astype(np.float64),
                          b.astype(np.float64))
    ilu = G.Ilu(gpu_ctx, rowp, cols)
    d_lu, d_b = dev(lu), dev(b)
    d_t, d_x = torch.zeros_like(d_b), torch.zeros_like(d_b)
    got = []
    for _ in range(3):
        ilu.apply(d_lu, d_b, d_t, d_x)
        gpu_ctx.sync()
        got.append(host(d_x).copy())
    # x may be the right-hand side's own memory
    d_in = d_b.clone()
    torch.cuda.synchronize()
    ilu.apply(d_lu, d_in, d_t, d_in)
    gpu_ctx.sync()
    got.append(host(d_in).copy())
    ilu.close()
    # the sums do not depend on the order in which rows become ready
    for g in got[1:]:
        assert np.array_equal(g.view(np.uint8), got[0].view(np.uint8))
    # |L^-1|, |U^-1| <= 2 in the max norm and at most 6 * 2,000 terms a sum:
    # a forward error of a few hundred roundings
    eps = np.finfo(dtype).eps
    assert np.abs(got[0] - x_o).max() <= 400 * eps * np.abs(x_o).max()
