"""The kernel timings take the launches of a solve: below 769 slices of 64 nodes a workgroup per
slice, above a wavefront per slice of each of the 8 XCDs' ranges."""
import pytest

import pfem_amd
from pfem_amd import meshgen as mg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,nodes,precision", [(2, 5000, "fp64"), (2, 50000, "fp64"), (2, 5000, "mixed"),
                                                 (3, 8000, "mixed")])
def test_residual_takes_a_v_cycles_launch(ctx, dim, nodes, precision):
    mesh = (mg.column_2d_nodes if dim == 2 else mg.column_3d_nodes)(nodes)
    print(f"[bench kernels] {dim}D N={mesh.n_nodes} {precision}", flush=True)
    q = mg.pspg_hydrostatic(mesh)
    c = pfem_amd.Case(ctx, dim, kind="PSPG", precision=precision, precond="amg")
    c.set_mesh(mesh)
    c.assemble(1e-3, q_prev=q, q_iter=q)
    k = c.bench_kernels(5)
    slices = -(-mesh.n_nodes // 64)
    assert k["amg_res0_blocks"] == (slices if slices <= 768 else 8 * -(-(-(-slices // 8)) // 4))
    assert k["amg_res0_us"] > 0 and k["kry_v_us"] > 0
    c.close()
