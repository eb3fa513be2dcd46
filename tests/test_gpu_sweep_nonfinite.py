"""Infinities and NaN in the triangular sweeps over row groups
(trsv_group_kernel): they reach the rows that depend on them and no others,
as in the level-by-level sweeps."""
import numpy as np
import pytest

import gpu_fem_amd as G
from gpu_helpers import dev, host
from test_gpu_sweep_groups import factors

pytestmark = pytest.mark.gpu

N = 1600  # above the sizes swept by one workgroup


def chains(length):
    """N rows in independent chains: several chains share a group record."""
    import scipy.sparse as sp

    i = np.arange(N - 1)
    i = i[i % length != length - 1]
    m = sp.csr_matrix((np.ones(2 * len(i) + N),
                       (np.r_[i, i + 1, np.arange(N)], np.r_[i + 1, i, np.arange(N)])), shape=(N, N))
    m.sort_indices()
    return m.indptr.astype(np.int32), m.indices.astype(np.int32)


def sweep(ctx, rowp, cols, lu, b):
    import torch

    ilu = G.Ilu(ctx, rowp, cols)
    d_b = dev(b)
    d_t, d_x = torch.zeros_like(d_b), torch.zeros_like(d_b)
    ilu.apply(dev(lu), d_b, d_t, d_x)
    ctx.sync()
    ilu.close()
    return host(d_x)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("where", ["rhs", "block", "diagonal"])
@pytest.mark.parametrize("length", [2, 4, 8])
def test_independent_rows_keep_their_values(gpu_ctx, length, where, dtype, monkeypatch):
    print(f"[gpu] non-finite sweeps chains of {length} {where} {np.dtype(dtype).name}", flush=True)
    rowp, cols = chains(length)
    lu = factors(rowp, cols, 1).astype(dtype)
    b = np.random.default_rng(2).standard_normal(6 * N).astype(dtype)
    clean = sweep(gpu_ctx, rowp, cols, lu, b)
    assert np.isfinite(clean).all()
    rows = np.repeat(np.arange(N), np.diff(rowp))
    # one value in one row of every eighth chain: of several groups in a
    # record (chains of 2 and 4) one or more stay clean
    hit = np.arange(0, N, 8 * length) + 1
    hit = hit[:len(hit) // 2 * 2]
    bad = np.array([np.inf, np.nan])[np.arange(len(hit)) % 2].astype(dtype)
    if where == "rhs":
        b[6 * hit + hit // length % 6] = bad
    else:
        j = hit - 1 if where == "block" else hit
        at = np.array([np.nonzero((rows == i) & (cols == k))[0][0] for i, k in zip(hit, j)])
        lu.reshape(-1, 6, 6)[at, 2, 3 if where == "block" else 2] = bad
    got = sweep(gpu_ctx, rowp, cols, lu, b)
    monkeypatch.setenv("GPUFEM_TRSV", "level")
    want = sweep(gpu_ctx, rowp, cols, lu, b)
    # the chains without such a value: the same bits as without any
    other = np.repeat(~np.isin(np.arange(N) // length, hit // length), 6)
    assert np.array_equal(got[other], clean[other])
    # the others: the same entries infinite and NaN, the finite ones as in the
    # sums of the sweeps' own tests
    assert not np.isfinite(want).all()
    for f in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(f(got), f(want))
    ok = np.isfinite(want)
    assert np.abs(got[ok] - want[ok]).max() <= 400 * np.finfo(dtype).eps * np.abs(want[ok]).max()
