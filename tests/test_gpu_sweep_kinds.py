"""Each kind of triangular sweep against the oracle's, chosen by GPUFEM_TRSV
and named by the analysis (gf_ilu_sweep_info), so that every case runs the
kernel it is meant for; and the kind that the pattern alone chooses."""
import numpy as np
import pytest

import gpu_fem_amd as G
import oracle
from gpu_fem_amd import meshes as M
from gpu_helpers import dev, host
from test_gpu_sweep_groups import CASES, factors, pattern

pytestmark = pytest.mark.gpu


def lu_pattern():
    """Complete block LU of a wingbox: U rows of up to 250 blocks."""
    m = M.wingbox(nc=24, nh=4, nsb=4, nribs=8, seed=5)
    rp, cp = G.node_graph(m.conn, m.nnodes)
    krp, kcp = G.pattern_permute(rp, cp, G.amd_order(rp, cp))
    return G.iluk_symbolic(krp, kcp, 1 << 29)[:2]


def make(kind, n):
    return lu_pattern() if kind == "wingbox" else pattern(n, kind, seed=n)


def check(ctx, rowp, cols, dtype, want):
    import torch

    n = len(rowp) - 1
    lu = factors(rowp, cols, n + 1).astype(dtype)
    b = np.random.default_rng(n + 2).standard_normal(6 * n).astype(dtype)
    x_o = oracle.bsr_trsv(rowp, cols, lu.astype(np.float64), b.astype(np.float64))
    ilu = G.Ilu(ctx, rowp, cols)
    assert ilu.sweep_info()["kind"] == want
    d_lu, d_b = dev(lu), dev(b)
    d_t, d_x = torch.zeros_like(d_b), torch.zeros_like(d_b)
    got = []
    for _ in range(2):
        ilu.apply(d_lu, d_b, d_t, d_x)
        ctx.sync()
        got.append(host(d_x).copy())
    ilu.close()
    assert np.array_equal(got[1].view(np.uint8), got[0].view(np.uint8))
    # as in the tests of the row groups: the factors' inverses are bounded
    assert np.abs(got[0] - x_o).max() <= 400 * np.finfo(dtype).eps * np.abs(x_o).max()


# rows: one pass of 64 blocks, the pass next to the diagonal after others
# (65 blocks and more), several passes
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("mode", ["rows", "groups"])
@pytest.mark.parametrize("kind,n", CASES + [("dense", 65), ("dense", 66), ("dense", 200), ("wingbox", 0)])
def test_chosen_kind(gpu_ctx, kind, n, mode, dtype, monkeypatch):
    print(f"[gpu] sweeps by {mode} {kind} n={n} {np.dtype(dtype).name}", flush=True)
    monkeypatch.setenv("GPUFEM_TRSV", "syncfree" if mode == "rows" else mode)
    check(gpu_ctx, *make(kind, n), dtype, mode)


@pytest.mark.parametrize("kind,n,want", [("chain", 1300, "small"), ("chain", 1301, "groups"), ("dense", 9, "small"),
                                         ("dense", 10, "groups"), ("random", 400, "rows"), ("band", 333, "groups"),
                                         ("wingbox", 0, "groups")])
def test_kind_by_the_pattern(gpu_ctx, kind, n, want):
    print(f"[gpu] sweep kind by the pattern {kind} n={n}", flush=True)
    check(gpu_ctx, *make(kind, n), np.float64, want)


@pytest.mark.parametrize("rowp,cols", [
    ([0, 2, 4], [1, 0, 0, 1]),       # not sorted
    ([0, 2, 4], [0, 0, 0, 1]),       # a column twice
    ([0, 2, 4], [0, 2, 0, 1]),       # out of range
    ([0, 2, 4], [-1, 0, 0, 1]),
    ([0, 1, 3], [1, 0, 1]),          # no diagonal block
    ([0, 0, 1], [1]),                # an empty row
    ([0, 1, 1], [0]),
])
def test_refused_patterns(gpu_ctx, rowp, cols):
    print(f"[gpu] refused pattern {rowp} {cols}", flush=True)
    with pytest.raises(G.GfError) as e:
        G.Ilu(gpu_ctx, np.array(rowp, np.int32), np.array(cols, np.int32))
    assert e.value.code == -1 and "ilu_create: row" in str(e.value)
