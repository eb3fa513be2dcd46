"""Element kernels that take four elements a wavefront, at element counts
around multiples of four (the last wavefront's blocks past the last element
are idle), on warped elements whose thickness, modulus and offset differ.

Tolerances as for the other element kernels: K 1e-12 per entry against
sqrt(|K_ii| |K_jj|), residual 1e-12 of its largest entry, energy 1e-12
relative."""
import ctypes

import numpy as np
import pytest

import gpu_fem_amd as G
import oracle
from gpu_fem_amd import meshes as M
from gpu_helpers import block_diag_scale, dev, host, max_rel_scaled, oracle_problem

pytestmark = pytest.mark.gpu


def strip(nelems, seed):
    m = M.plate(nelems, 1, 0.3 * nelems, 0.4, thick=0.01)
    assert m.nelems == nelems
    rng = np.random.default_rng(seed)
    m.xpts[:, :2] += rng.uniform(-0.04, 0.04, (m.nnodes, 2))
    m.xpts[:, 2] = rng.uniform(-0.03, 0.03, m.nnodes)
    m.data[:, 0] *= rng.uniform(0.5, 2.0, nelems)
    m.data[:, 1] = rng.uniform(0.1, 0.4, nelems)
    m.data[:, 2] = rng.uniform(0.005, 0.02, nelems)
    m.data[:, 3] = rng.uniform(-0.4, 0.4, nelems)
    return m


@pytest.mark.parametrize("nelems", [1, 2, 3, 4, 5, 8, 9, 15, 17])
@pytest.mark.parametrize("nonlinear", [False, True])
def test_element_counts(gpu_ctx, nelems, nonlinear):
    import torch

    print(f"[gpu] element kernels n={nelems} nonlinear={nonlinear}", flush=True)
    m = strip(nelems, nelems)
    s = oracle_problem(m, "rcm", 0)
    nnzb = int(s["krp"][-1])
    u = 1e-2 * np.random.default_rng(nelems).standard_normal(6 * m.nnodes)
    xyz = np.asarray(m.xpts).reshape(-1, 3)
    if nonlinear:
        kv_o, res_o, e_o = oracle.assemble_tangent(
            m.conn, m.xpts, m.data, s["emap"], s["perm"], nnzb, u)
    else:
        kv_o, res_o = oracle.assemble_jacobian(
            m.conn, m.xpts, m.data, s["emap"], s["perm"], nnzb, vars=u)
        e_o = sum(oracle.element(xyz[c], u.reshape(-1, 6)[c].ravel(),
                                 m.data[i])[2] for i, c in enumerate(m.conn))
    scale = block_diag_scale(s["krp"], s["kcp"], kv_o)
    d_conn, d_x = dev(m.conn, np.int32), dev(m.xpts, np.float64)
    d_data, d_u = dev(m.data, np.float64), dev(u)
    d_map, d_perm = dev(s["emap"]), dev(s["perm"])
    L = G.lib()

    def check(kv, res):
        gpu_ctx.sync()
        if kv is not None:
            assert max_rel_scaled(host(kv), kv_o, scale) <= 1e-12
        assert np.abs(host(res) - res_o).max() <= 1e-12 * np.abs(res_o).max()

    def zeros():
        return (torch.zeros(36 * nnzb, dtype=torch.float64, device="cuda"),
                torch.zeros(6 * m.nnodes, dtype=torch.float64, device="cuda"))

    e = torch.zeros(1, dtype=torch.float64, device="cuda")
    plan = ctypes.c_void_p()
    gpu_ctx.check(L.gf_asm_plan_create(
        gpu_ctx.h, m.nelems, m.nnodes,
        G.ptr(np.ascontiguousarray(m.conn, np.int32)),
        G.ptr(np.ascontiguousarray(s["emap"], np.int32)), nnzb,
        ctypes.byref(plan)))
    k, r = zeros()
    kc, rc = (t + 3.0 for t in zeros())  # colour order: no zeroing needed
    if nonlinear:
        gpu_ctx.check(L.gf_assemble_tangent_mitc4_f64(
            gpu_ctx.h, m.nelems, m.nnodes, G.ptr(d_conn), G.ptr(d_x),
            G.ptr(d_u), G.ptr(d_data), G.ptr(d_map), G.ptr(d_perm), G.ptr(k),
            G.ptr(r), G.ptr(e)))
        gpu_ctx.check(L.gf_assemble_tangent_colored_f64(
            gpu_ctx.h, plan, G.ptr(d_conn), G.ptr(d_x), G.ptr(d_u),
            G.ptr(d_data), G.ptr(d_map), G.ptr(d_perm), G.ptr(kc), G.ptr(rc)))
    else:
        gpu_ctx.check(L.gf_assemble_jacobian_mitc4_f64(
            gpu_ctx.h, m.nelems, m.nnodes, G.ptr(d_conn), G.ptr(d_x),
            G.ptr(d_u), G.ptr(d_data), G.ptr(d_map), G.ptr(d_perm), G.ptr(k),
            G.ptr(r)))
        gpu_ctx.check(L.gf_assemble_jacobian_colored_f64(
            gpu_ctx.h, plan, G.ptr(d_conn), G.ptr(d_x), G.ptr(d_u),
            G.ptr(d_data), G.ptr(d_map), G.ptr(d_perm), G.ptr(kc), G.ptr(rc)))
        gpu_ctx.check(L.gf_energy_mitc4_f64(
            gpu_ctx.h, m.nelems, G.ptr(d_conn), G.ptr(d_x), G.ptr(d_u),
            G.ptr(d_data), G.ptr(e)))
        r1 = zeros()[1]
        gpu_ctx.check(L.gf_assemble_residual_mitc4_f64(
            gpu_ctx.h, m.nelems, m.nnodes, G.ptr(d_conn), G.ptr(d_x),
            G.ptr(d_u), G.ptr(d_data), G.ptr(d_perm), G.ptr(r1)))
        check(None, r1)
        # no displacements: the same K, no residual
        kn, rn = zeros()
        gpu_ctx.check(L.gf_assemble_jacobian_mitc4_f64(
            gpu_ctx.h, m.nelems, m.nnodes, G.ptr(d_conn), G.ptr(d_x), None,
            G.ptr(d_data), G.ptr(d_map), G.ptr(d_perm), G.ptr(kn), G.ptr(rn)))
        gpu_ctx.sync()
        assert max_rel_scaled(host(kn), kv_o, scale) <= 1e-12
        assert not host(rn).any()
    check(k, r)
    check(kc, rc)
    assert abs(host(e)[0] - e_o) <= 1e-12 * abs(e_o)
    L.gf_asm_plan_destroy(plan)
