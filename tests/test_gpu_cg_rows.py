"""The conjugate gradients of the heat and fractional-step solvers where their products' row split
changes: node counts that leave a workgroup's last lane groups empty, one workgroup, and more nodes
than the products' grid covers in one round (32,768 in 3D), against the oracle.

Tolerances: both sides solve to a relative residual of 1e-13; the condition numbers (under 1e3 for
the heat system with its mass term, 1e4 for the pressure system) carry that to 1e-9 of the largest
value of the temperatures and velocities and 1e-8 of the pressures."""
import numpy as np
import pytest

import pfem_amd
from oracle import oracle as O
from pfem_amd import _lib
from test_gpu_fracstep import closed_box, frac_case, gvec
from test_gpu_heat import block_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,n", [(2, 5), (2, 16), (3, 4), (3, 33)])
def test_heat_rows_match_oracle(ctx, dim, n):
    mesh, fac, out, kinds, left = block_case(dim, n)
    print(f"[cg rows] heat {dim}D N={mesh.n_nodes}", flush=True)
    T = 300.0 + np.random.default_rng(3).normal(scale=10.0, size=mesh.n_nodes)
    Tbc = np.zeros(mesh.n_nodes)
    Tbc[left] = 400.0
    mat = dict(rho=900.0, cv=2000.0, k=5.0, h=30.0, Tinf=290.0, epsRad=0.7)
    case = pfem_amd.HeatEqIncompNewton(ctx, dim, krylov_rtol=1e-13, **mat)
    case.set_mesh(mesh)
    case.set_state(T)
    case.set_facets(fac, out, kinds & ~np.uint8(O.HEAT_Q))
    case.set_dirichlet_T(Tbc)
    hc = O.HeatCase(facets=fac, facet_out=out, facet_kind=kinds & ~np.uint8(O.HEAT_Q), **mat)
    assert case.solve(5.0), case.last_stats
    st, _, _ = O.heat_step(mesh, T, Tbc=Tbc, hc=hc, dt=5.0, rtol=1e-13)
    assert st == 0
    assert np.abs(case.get_state() - T).max() <= 1e-9 * np.abs(T).max()
    case.close()


@pytest.mark.parametrize("dim,n", [(2, 5), (3, 4), (3, 33)])
def test_frac_rows_match_oracle(ctx, dim, n):
    mesh, _ = closed_box(dim, n=n)
    d, N = dim, mesh.n_nodes
    print(f"[cg rows] frac {dim}D N={N}", flush=True)
    kw = dict(rho=1000.0, mu=1e-3, residual="U", max_iter=3)
    q_ref, pos_ref, g = np.zeros((d + 1) * N), mesh.pos.copy(), gvec(dim)
    st_ref, s_ref = O.frac_step(mesh, pos_ref, q_ref, g=g, dt=1e-2, gamma_fs=0.0, **kw)
    c = frac_case(ctx, dim, mesh, body_force=list(g), gammaFS=0.0, krylov_rtol=1e-13, **kw)
    rc, st = c.step(1e-2)
    assert st_ref == 0 and rc == _lib.PFEM_OK and st["picard_iters"] == s_ref["picard_iters"]
    q = c.get_state()
    assert np.abs(q[: d * N] - q_ref[: d * N]).max() < 1e-9 * np.abs(q_ref[: d * N]).max()
    assert np.ptp(q[d * N:] - q_ref[d * N:]) < 1e-8 * np.abs(q_ref[d * N:]).max()
    c.close()
