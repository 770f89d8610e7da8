"""The CFL time step of the weakly compressible solver.

A run restarted from its saved states and positions goes on with the bits of an uninterrupted one:
the minimum that the step's last pass leaves equals the CFL pass over the same state, exactly.  (The
meshes are those at the limits of the step's tiles.)

One element of integer coordinates at rest, against longdouble: edges, areas and det J are whole
numbers below 2^53 and exact, so he = 2 r_in carries the roundings of its square roots (an ulp,
2.3e-16 each, of which he sees their weighted mean), three sums and a division, and dt half of two
products' and a division's, half of c^2's and its own square root: under 1e-15 together."""
import numpy as np
import pytest

import pfem_amd
from pfem_amd import meshgen as mg
from test_gpu_wc_tiles import CASES, K0, K0P, MU, RS

pytestmark = pytest.mark.gpu


def case_of(ctx, mesh, state):
    c = pfem_amd.Case(ctx, mesh.dim, kind="WC", mu=MU, K0=K0, K0p=K0P, rho_star=RS, wc_state=state)
    c.set_mesh(mesh)
    return c


@pytest.mark.parametrize("state", ["fp64", "fp32"])
@pytest.mark.parametrize("name", list(CASES))
def test_restart_takes_the_same_steps(ctx, name, state):
    mesh = CASES[name]()
    print(f"[wc cfl] {name} {state} N={mesh.n_nodes}", flush=True)
    v, p, rho, a = mg.wc_tait_hydrostatic(mesh, K0=K0, K0p=K0P, rho_star=RS)
    v = v + 0.02 * np.random.default_rng(5).standard_normal(v.shape) * ((mesh.flags & mg.BOUND) == 0)
    one, two = case_of(ctx, mesh, state), case_of(ctx, mesh, state)
    one.set_state(np.concatenate([v.reshape(-1), p, rho, a.reshape(-1)]))
    for k in range(4):
        dt = one.wc_next_dt(0.5, 1.0)
        two.set_state(one.get_state())
        two.set_positions(one.get_positions())
        assert two.wc_next_dt(0.5, 1.0) == dt, k
        one.wc_step(dt)
        two.wc_step(dt)
        assert np.array_equal(one.get_state(), two.get_state()), k
        assert np.array_equal(one.get_positions(), two.get_positions()), k
    one.close()
    two.close()


@pytest.mark.parametrize("dim", [2, 3])
def test_single_elements_against_longdouble(ctx, dim):
    rng = np.random.default_rng(dim)
    L = np.longdouble
    print(f"[wc cfl] elements {dim}D", flush=True)
    worst = 0.0
    for _ in range(60):
        x = rng.integers(0, 1000, (dim + 1, dim)).astype(float)
        e = x[1:] - x[0]
        dj = np.round(np.linalg.det(e))
        if abs(dj) < 1000 ** dim / 50:
            continue
        if dj < 0:
            x[[1, 2]] = x[[2, 1]]
        mesh = mg.PfemMesh(dim, np.ascontiguousarray(x.T), np.arange(dim + 1, dtype=np.int32)[None], np.zeros(dim + 1, np.uint8),
                           1.0, surface=np.full(dim + 1, 1e3))
        c = case_of(ctx, mesh, "fp64")
        N = dim + 1
        c.set_state(np.concatenate([np.zeros(dim * N), np.zeros(N), np.full(N, RS), np.zeros(dim * N)]))
        dt = c.wc_next_dt(0.5, 1e9)
        c.close()
        xl = x.astype(L)
        if dim == 2:
            per = sum(np.sqrt(((xl[i] - xl[j]) ** 2).sum()) for i, j in ((0, 1), (1, 2), (0, 2)))
            he = 2 * (abs(L(dj)) / 2) / (per / 2)
        else:
            area = lambda o, i, j: np.sqrt((np.cross(xl[i] - xl[o], xl[j] - xl[o]) ** 2).sum()) / 2
            he = 2 * 3 * (abs(L(dj)) / 6) / (area(0, 1, 2) + area(0, 1, 3) + area(0, 2, 3) + area(1, 2, 3))
        alpha = L(MU) / L(RS)
        ref = np.sqrt(L(0.25) * he * he / max(L(K0) / L(RS), 4 * alpha * alpha / (he * he)))
        worst = max(worst, float(abs(L(dt) - ref) / ref))
    print(f"[wc cfl] worst relative difference {worst:.2e}", flush=True)
    assert worst <= 1e-15, worst
