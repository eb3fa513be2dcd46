"""Numeric ILU row kernels on patterns at their edges: windows of pivots that
wrap and that do not divide the pivot count, rows of one block, rows whose
whole U part lies at the ends of their cache lines, patterns that are not
symmetric, and rows of more blocks than a workgroup has threads."""
import numpy as np
import pytest

import gpu_fem_amd as G
import oracle
from gpu_helpers import dev, host
from test_gpu_sweep_groups import pattern

pytestmark = pytest.mark.gpu


def matrix(rowp, cols, seed):
    """Block rows dominated by their diagonal entries (ILU without pivoting
    is well conditioned)."""
    rng = np.random.default_rng(seed)
    n = len(rowp) - 1
    rows = np.repeat(np.arange(n), np.diff(rowp))
    v = rng.uniform(-1.0, 1.0, (len(cols), 6, 6))
    d = np.nonzero(rows == cols)[0]
    for a in range(6):
        v[d, a, a] = 12.0 * np.diff(rowp) + rng.uniform(1.0, 2.0, n)
    return v.ravel()


CASES = [("dense", 1), ("dense", 2), ("dense", 3), ("dense", 9),
         ("dense", 70), ("chain", 50), ("band", 200), ("forest", 300),
         ("random", 300), ("lower", 100), ("chained", 250), ("dense", 530)]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind,n", CASES)
def test_row_kernels_agree(gpu_ctx, kind, n, dtype, monkeypatch):
    """Rows in LDS, rows with their pivots applied in runs (windows of 2, 5, 7
    and 8) and one pivot at a time do the same operations in the same order:
    the factors agree bit for bit, and with the oracle's to rounding."""
    print(f"[gpu] ilu rows {kind} n={n} {np.dtype(dtype).name}", flush=True)
    rowp, cols = pattern(n, kind, seed=n)
    a = matrix(rowp, cols, n).astype(dtype)
    ilu = G.Ilu(gpu_ctx, rowp, cols)

    def factor():
        d = dev(a)
        ilu.factor(d)
        gpu_ctx.sync()
        return host(d)

    got = {"rows in LDS": factor()}
    monkeypatch.setenv("GPUFEM_ILU_GLOBAL", "1")
    for nbatch in (2, 5, 7, 8):
        monkeypatch.setenv("GPUFEM_ILU_BATCH_N", str(nbatch))
        got[f"window {nbatch}"] = factor()
    monkeypatch.delenv("GPUFEM_ILU_BATCH_N")
    monkeypatch.setenv("GPUFEM_ILU_GLOBAL_KERNEL", "pivot")
    ref = factor()
    ilu.close()
    for name, lu in got.items():
        assert np.array_equal(lu.view(np.uint8), ref.view(np.uint8)), name
    if n <= 300:
        lu_o, st = oracle.bsr_ilu(rowp, cols, a.astype(np.float64))
        assert st == 0
        # growth below 2 in a diagonally dominant elimination: a few roundings
        # per term of sums of at most 6 n terms
        eps = np.finfo(dtype).eps
        assert np.abs(ref - lu_o).max() <= 100 * eps * np.abs(lu_o).max()
