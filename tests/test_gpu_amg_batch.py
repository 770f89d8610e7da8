"""Multigrid steps in a batch large enough for the coarse levels' residual and restriction to take a
launch each (over 2,048 aggregates in all) against the same step alone, where they share one: the
same bits, with hierarchies in FP64, in FP64 with FP32 level-0 values, and wholly in FP32."""
import numpy as np
import pytest

import pfem_amd
from pfem_amd import meshgen as mg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,nodes,precision,copies", [(2, 20000, "fp64", 16), (3, 60000, "mixed", 24),
                                                        (3, 60000, "mixed_all_fp32", 24)])
def test_large_batch_equals_alone(ctx, dim, nodes, precision, copies, monkeypatch):
    if precision == "mixed_all_fp32":
        monkeypatch.setenv("PFEM_AMG_FP32", "1")
    mesh = (mg.column_2d_nodes if dim == 2 else mg.column_3d_nodes)(nodes)
    print(f"[amg batch] {copies} x {dim}D N={mesh.n_nodes} {precision}", flush=True)
    q = mg.pspg_hydrostatic(mesh)
    dt = 1e-3 if dim == 2 else 5e-4

    def make():
        c = pfem_amd.Case(ctx, dim, kind="PSPG", precision=precision[:5] if dim == 3 else precision, precond="amg",
                          krylov_rtol=1e-8, max_iter=2, min_res=1e-3)
        c.set_mesh(mesh)
        c.set_state(q)
        return c

    one = make()
    rc, st = one.pspg_step(dt)
    assert rc == 0, st
    cases = [make() for _ in range(copies)]
    status, stats = pfem_amd.batch_step(ctx, cases, [dt] * copies)
    assert list(status) == [0] * copies, stats
    for c in cases:
        assert np.array_equal(c.get_state(), one.get_state()) and np.array_equal(c.get_positions(), one.get_positions())
        c.close()
    one.close()
