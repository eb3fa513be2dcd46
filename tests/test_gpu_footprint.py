"""Admission of the serving loop counts what the ILU analysis of a request
allocates: the records of its row groups, or the row descriptors and chunks of
a pattern without groups, not a bound of both."""
import ctypes

import pytest

import gpu_fem_amd as G
from gpu_fem_amd import meshes as M

pytestmark = pytest.mark.gpu


def block_class(b):
    """Size of a cached device block: 4 KiB, then quarters of powers of two."""
    if b <= 4096:
        return 4096
    q = 1 << (b.bit_length() - 3)
    return -(-b // q) * q


@pytest.mark.parametrize("nx,fill", [(20, 3), (45, 12)])
def test_peak_bytes_of_row_groups(gpu_ctx, nx, fill, monkeypatch):
    print(f"[gpu] footprint plate {nx} ILU({fill})", flush=True)
    m = M.plate(nx, nx, thick=0.01)
    opts = dict(reorder=2, lev_fill=fill, restart=60, rtol=1e-8, max_iters=4000)
    peak, info = {}, {}
    for mode in ("syncfree", "groups"):
        monkeypatch.setenv("GPUFEM_TRSV", mode)
        p = G.Problem(gpu_ctx, m, **opts)
        c = [ctypes.c_int() for _ in range(3)]
        G.check(G.lib().gf_ilu_sweep_info(p.ilu_handle(), *[ctypes.byref(v) for v in c]))
        info[mode] = [v.value for v in c]
        p.close()
        srv = G.Server(budget_gb=10.0, slots=1)
        assert srv.submit(0, m, **opts) == 0
        srv.drain()
        peak[mode] = srv.stats()["peak_bytes"]
        srv.close()
    assert info["syncfree"][0] == 2 and info["groups"][0] == 3
    n = m.nnodes
    rows = 2 * block_class(4 * (n + 1)) + 2 * block_class(16 * n)
    records = sum(block_class(32 * k) + block_class(384 * k) for k in info["groups"][1:])
    assert peak["groups"] - peak["syncfree"] == records - rows
