"""The tile passes of the weakly compressible step against the oracle where their tiles are at
their limits: node counts around whole tiles, nodes numbered at random (a tile then refers to
more nodes than it stages, so elements are visited through memory), a node with more elements
than a tile's staged visit words, nodes in no element, and 3D cases on both sides of the size
(16,384 nodes) up to which tiles are small.

Tolerance: the FP64 step differs from the oracle by the rounding of its sums and of a handful of
products per element, a few hundred ulp (1e-13) of the largest term; the pressure terms that
cancel in an acceleration are at most ~1e3 times it on these meshes, so 1e-10 of each field."""
import numpy as np
import pytest

import pfem_amd
from oracle import oracle as O
from pfem_amd import meshgen as mg

pytestmark = pytest.mark.gpu

K0, K0P, RS, MU = 2.2e6, 7.0, 1000.0, 1e-3


def renumber(mesh, seed):
    """The same mesh with its nodes in random order."""
    perm = np.random.default_rng(seed).permutation(mesh.n_nodes)  # old -> new
    inv = np.argsort(perm)
    return mg.PfemMesh(mesh.dim, np.ascontiguousarray(mesh.pos[:, inv]), perm[mesh.conn].astype(np.int32),
                       mesh.flags[inv], mesh.h, surface=mesh.surface[inv])


def fan(n):
    """n triangles around one node, and one node in no element."""
    t = 2 * np.pi * np.arange(n) / n
    pos = np.hstack([[[0.0], [1.0]], np.stack([np.cos(t), 1.0 + np.sin(t)]), [[5.0], [5.0]]])
    k = np.arange(n)
    conn = np.stack([np.zeros(n, int), 1 + k, 1 + (k + 1) % n], axis=1).astype(np.int32)
    return mg.PfemMesh(2, pos, conn, np.zeros(n + 2, np.uint8), 0.1, surface=np.full(n + 2, 2.0))


def strip(n_nodes):
    """A 2D strip, two nodes wide, with exactly n_nodes nodes (the last ones in no element)."""
    nx = n_nodes // 2 - 1
    m = mg.tank_2d(h=0.1, size=(0.1 * nx, 0.1), fill=1.0, seed=4)
    extra = n_nodes - m.n_nodes
    pos = np.hstack([m.pos, 7.0 + np.zeros((2, extra))])
    return mg.PfemMesh(2, pos, m.conn, np.concatenate([m.flags, np.zeros(extra, np.uint8)]), m.h,
                       surface=np.concatenate([m.surface, np.full(extra, 8.0)]))


CASES = {
    "2d_one_tile": lambda: strip(128), "2d_tile_plus_one": lambda: strip(129), "2d_tile_less_one": lambda: strip(127),
    "2d_random_order": lambda: renumber(mg.tank_nodes(2, 3000), 1), "2d_fan_1200": lambda: fan(1200),
    "3d_small": lambda: mg.tank_3d(h=0.5, size=(1.0, 1.0, 1.0), fill=1.0),
    "3d_random_order": lambda: renumber(mg.tank_nodes(3, 4000), 2),
    "3d_large_tiles_random_order": lambda: renumber(mg.tank_nodes(3, 20000), 2),
}


@pytest.mark.parametrize("name", list(CASES))
def test_wc_tile_limits_match_oracle(ctx, name):
    mesh = CASES[name]()
    d, N = mesh.dim, mesh.n_nodes
    print(f"[wc tiles] {name} N={N} E={mesh.n_elems}", flush=True)
    v, p, rho, a = mg.wc_tait_hydrostatic(mesh, K0=K0, K0p=K0P, rho_star=RS)
    v = v + 0.02 * np.random.default_rng(5).standard_normal(v.shape) * ((mesh.flags & mg.BOUND) == 0)
    c = pfem_amd.Case(ctx, d, kind="WC", mu=MU, K0=K0, K0p=K0P, rho_star=RS)
    c.set_mesh(mesh)
    c.set_state(np.concatenate([v.reshape(-1), p, rho, a.reshape(-1)]))
    pos = mesh.pos.reshape(-1).copy()
    vo, po, ro, ao = v.reshape(-1).copy(), p.copy(), rho.copy(), a.reshape(-1).copy()
    for _ in range(2):
        dt = O.wc_next_dt(mesh, pos, vo, po, ro, mu=MU, K0=K0, K0p=K0P, security_coeff=0.5, max_dt=1e-3)
        assert c.wc_next_dt(0.5, 1e-3) == pytest.approx(dt, rel=1e-12)
        O.wc_step(mesh, pos, vo, po, ro, ao, dt, mu=MU, K0=K0, K0p=K0P, rho_star=RS)
        c.wc_step(dt)
    s = c.get_state()
    for got, ref in ((s[:d * N], vo), (s[d * N:(d + 1) * N], po), (s[(d + 1) * N:(d + 2) * N], ro),
                     (s[(d + 2) * N:], ao), (c.get_positions().reshape(-1), pos)):
        assert np.abs(got - ref).max() <= 1e-10 * max(np.abs(ref).max(), 1e-3)
    c.close()
