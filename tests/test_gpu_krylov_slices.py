"""BiCGSTAB over the 64-node slices of the system where their split can go wrong: a single slice,
whole slices and one node more, one slice per XCD and one more, and both sides of the number of
slices up to which a workgroup's wavefronts share a slice (768) — with block Jacobi and with
multigrid, in FP64 and with FP32 inner solves — against the oracle's system.

Tolerance: the solver stops on its own true residual at 1e-8 ||b||; the oracle's residual of the
same x differs by the rounding of the two assemblies (under 1e-12 of each entry, which times the
ratio of |A| |x| to |b|, at most 1e3 on these meshes, is 1e-9), so 2e-8."""
import numpy as np
import pytest

import pfem_amd
from oracle import oracle as O
from pfem_amd import meshgen as mg

pytestmark = pytest.mark.gpu


def column(dim, n_nodes):
    """A column of liquid with exactly n_nodes nodes (the last ones in no element)."""
    make = mg.column_2d_nodes if dim == 2 else mg.column_3d_nodes
    target = n_nodes
    while (m := make(target, h=0.01, seed=2)).n_nodes > n_nodes:
        target = int(0.95 * target)
    extra = n_nodes - m.n_nodes
    assert 0 <= extra < n_nodes
    pos = np.hstack([m.pos, 7.0 + np.zeros((dim, extra))])
    return mg.PfemMesh(dim, pos, m.conn, np.concatenate([m.flags, np.zeros(extra, np.uint8)]), m.h,
                       surface=np.concatenate([m.surface, np.full(extra, 8.0)]))


@pytest.mark.parametrize("dim,n_nodes,precond,precision", [
    (2, 64, "jacobi", "fp64"), (2, 65, "jacobi", "mixed_ir"), (2, 512, "jacobi", "fp64"), (2, 513, "amg", "fp64"),
    (3, 128, "jacobi", "fp64"), (3, 129, "jacobi", "mixed_ir"), (3, 577, "jacobi", "mixed"),
    (2, 49152, "amg", "fp64"), (2, 49153, "amg", "fp64"), (3, 49152, "jacobi", "mixed_ir"),
    (3, 49153, "jacobi", "mixed_ir"), (3, 49153, "jacobi", "fp64"),
])
def test_solve_at_slice_limits(ctx, dim, n_nodes, precond, precision):
    mesh = column(dim, n_nodes)
    print(f"[slices] dim={dim} N={mesh.n_nodes} {precond} {precision}", flush=True)
    q = mg.pspg_hydrostatic(mesh)
    dt = 1e-3 if dim == 2 else 5e-4
    ref = O.pspg_assemble(mesh, q, q, dt=dt)
    A = ref.to_scipy()
    c = pfem_amd.Case(ctx, dim, kind="PSPG", precision=precision, krylov_rtol=1e-8, precond=precond)
    c.set_mesh(mesh)
    c.assemble(dt, q_prev=q, q_iter=q)
    first = None
    for _ in range(2):  # a second solve of the same system gives the same bits
        rc, x, st = c.solve(x0=np.zeros_like(q))
        assert rc == 0, st
        relres = np.linalg.norm(ref.b - A @ x) / np.linalg.norm(ref.b)
        assert relres <= 2e-8, (relres, st)
        assert first is None or np.array_equal(first, x)
        first = x
    c.close()
