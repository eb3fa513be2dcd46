"""Small systems: both sweeps by one workgroup (trsv_small_kernel), its rule's
edges, the short-vector kernels of GMRES, and small systems among others in
the batched serving engine."""
import numpy as np
import pytest

import gpu_fem_amd as G
import oracle
from gpu_fem_amd import meshes as M
from gpu_helpers import dev, host
from test_gpu_sweep_groups import factors, pattern

pytestmark = pytest.mark.gpu


def narrow(n, kind, seed):
    """At most eight blocks on either side of a row's diagonal."""
    import scipy.sparse as sp

    if kind == "band8":
        m = sp.diags([1.0] * 17, range(-8, 9), shape=(n, n))
    elif kind == "band9":  # one block too many: swept by the other kernels
        m = sp.diags([1.0] * 19, range(-9, 10), shape=(n, n))
    elif kind == "diagonal":  # one level, rows without dependencies
        m = sp.eye(n)
    elif kind == "chain":  # a level a row
        return pattern(n, "chain")
    else:  # sparse, not symmetric, rows of any length up to eight
        rng = np.random.default_rng(seed)
        m = sp.lil_matrix((n, n))
        for i in range(n):
            for lo, hi in ((0, i), (i + 1, n)):
                k = min(hi - lo, int(rng.integers(0, 9)))
                m[i, rng.choice(np.arange(lo, hi), k, replace=False)] = 1.0
            m[i, i] = 1.0
    m = sp.csr_matrix(m)
    m.sort_indices()
    return m.indptr.astype(np.int32), m.indices.astype(np.int32)


CASES = [("diagonal", 1), ("chain", 2), ("chain", 17), ("band8", 15),
         ("band8", 49), ("band9", 49), ("diagonal", 100), ("random", 16),
         ("random", 48), ("random", 333), ("band8", 1300), ("band8", 1301)]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind,n", CASES)
def test_small_sweeps_match_oracle(gpu_ctx, kind, n, dtype, monkeypatch):
    import torch

    print(f"[gpu] small sweeps {kind} n={n} {np.dtype(dtype).name}", flush=True)
    rowp, cols = narrow(n, kind, n)
    lu = factors(rowp, cols, n + 1).astype(dtype)
    b = np.random.default_rng(n + 2).standard_normal(6 * n).astype(dtype)
    x_o = oracle.bsr_trsv(rowp, cols, lu.astype(np.float64),
                          b.astype(np.float64))
    d_lu, d_b = dev(lu), dev(b)
    # tolerance as for the row-group sweeps of the same factors
    tol = 400 * np.finfo(dtype).eps * np.abs(x_o).max()
    for mode in ("small", "syncfree", None):  # None: by the rule
        if mode:
            monkeypatch.setenv("GPUFEM_TRSV", mode)
        else:
            monkeypatch.delenv("GPUFEM_TRSV")
        ilu = G.Ilu(gpu_ctx, rowp, cols)
        d_t, d_x = torch.zeros_like(d_b), torch.full_like(d_b, np.nan)
        got = []
        for _ in range(3):
            ilu.apply(d_lu, d_b, d_t, d_x)
            gpu_ctx.sync()
            got.append(host(d_x).copy())
        d_in = d_b.clone()  # x may be the right-hand side's own memory
        torch.cuda.synchronize()
        ilu.apply(d_lu, d_in, d_t, d_in)
        gpu_ctx.sync()
        got.append(host(d_in).copy())
        ilu.close()
        for g in got[1:]:
            assert np.array_equal(g.view(np.uint8), got[0].view(np.uint8))
        assert np.abs(got[0] - x_o).max() <= tol, mode


@pytest.mark.parametrize("precision", [0, 2], ids=["fp64", "fp32 ilu"])
def test_small_systems_in_the_batched_engine(gpu_ctx, precision, monkeypatch):
    """Plates swept by one workgroup next to one that is not, solved together:
    each result equals the solve alone (1e-10)."""
    monkeypatch.setenv("GPUFEM_SERVE_BATCH", "1")
    print(f"[gpu] small systems served, precision {precision}", flush=True)
    small = dict(reorder=0, lev_fill=0, restart=400, rtol=1e-9,
                 max_iters=4000, precision=precision)
    large = dict(small, reorder=2, lev_fill=3)
    reqs = [(M.plate(k, k, thick=0.01), small) for k in (3, 5, 7, 4)]
    reqs.insert(2, (M.plate(24, 24, thick=0.01), large))
    alone = []
    for m, o in reqs:
        p = G.Problem(gpu_ctx, m, **o)
        p.assemble()
        p.factor()
        x, info = p.solve()
        assert info.status == 0
        alone.append(x)
        p.close()
    srv = G.Server(budget_gb=50.0, slots=5)
    for i, (m, o) in enumerate(reqs):
        assert srv.submit(i, m, **o) == 0
    srv.drain()
    got = 0
    while True:
        r = srv.poll()
        if r is None:
            break
        rid, x, info, _ = r
        assert info.status == 0 and info.rel_resid <= 1e-9
        xa = alone[rid]
        assert np.linalg.norm(x - xa) <= 1e-10 * np.linalg.norm(xa), rid
        got += 1
    srv.close()
    assert got == len(reqs)
