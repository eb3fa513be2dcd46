"""Values into a wider block pattern: target rows around the workgroup's chunk,
source rows shorter and longer than the columns kept in LDS, empty rows, and
values whose address is a multiple of 8 bytes only."""
import numpy as np
import pytest

import gpu_fem_amd as G
from gpu_helpers import dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("n,src,tgt", [(1, 1, 1), (40, 3, 40), (127, 9, 127),
                                       (128, 64, 128), (130, 65, 129),
                                       (300, 100, 257), (300, 300, 300)])
def test_copy_rows(gpu_ctx, n, src, tgt, shift):
    import torch

    print(f"[gpu] copy pattern n={n} source {src} target {tgt} shift {shift}",
          flush=True)
    rng = np.random.default_rng(n + src)
    rows_s, rows_t = [], []
    for i in range(n):
        kt = int(rng.integers(0, tgt + 1)) if i else tgt
        t = np.sort(rng.choice(n, kt, replace=False))
        ks = min(kt, src if i == 0 else int(rng.integers(0, src + 1)))
        rows_t.append(t)
        rows_s.append(np.sort(rng.choice(t, ks, replace=False)))

    def csr(rows):
        return (np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32),
                np.concatenate(rows).astype(np.int32))

    rp, cp = csr(rows_s)
    trp, tcp = csr(rows_t)
    vals = rng.standard_normal((len(cp), 36))
    want = np.zeros((len(tcp), 36))
    for i in range(n):
        at = trp[i] + np.searchsorted(rows_t[i], rows_s[i])
        want[at] = vals[rp[i]:rp[i + 1]]
    pad = np.zeros(shift)
    d_v = dev(np.concatenate([pad, vals.ravel()]))
    d_t = torch.full((shift + want.size + 1,), np.nan, dtype=torch.float64,
                     device="cuda")
    d_rp, d_cp, d_trp, d_tcp = dev(rp), dev(cp), dev(trp), dev(tcp)
    gpu_ctx.check(G.lib().gf_bsr_copy_to_pattern(
        gpu_ctx.h, n, G.ptr(d_rp), G.ptr(d_cp), G.ptr(d_v[shift:]),
        G.ptr(d_trp), G.ptr(d_tcp), G.ptr(d_t[shift:])))
    gpu_ctx.sync()
    got = d_t.cpu().numpy()
    assert np.array_equal(got[shift:shift + want.size], want.ravel())
    assert np.isnan(got[:shift]).all() and np.isnan(got[-1])
