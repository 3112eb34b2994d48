"""GPU: how far one non-finite eddy viscosity reaches in the viscous residual of tets: its own cell (the d/dc
rows are dense), and at a neighbour the solution points on the lines of those flux points whose
interpolation row names the point.  The set is formed here from the mesh's tables."""

import numpy as np
import pytest

from cases import freestream, prim_to_cons, tet_box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,prec", [(1, "f32"), (1, "f64"), (2, "f32"), (2, "f64"), (3, "f64")])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_reach_of_a_non_finite_eddy_viscosity(order, prec, value):
    import torch
    from autoflowcfd_amd.device import DeviceMesh, bc_params_table
    print(f"[gpu] reach of a non-finite mu_t P{order} {prec} {value}", flush=True)
    dt = torch.float32 if prec == "f32" else torch.float64
    Q0 = freestream(0.15, 4.0)
    mesh = tet_box(2, seed=1)
    dm = DeviceMesh(mesh, order, dtype=dt, bc_params=bc_params_table(Q0))
    U = torch.as_tensor(prim_to_cons(Q0), dtype=dt, device="cuda").expand(mesh.n_cells, dm.ns, 5).contiguous()
    host = lambda x: x.cpu().numpy()  # noqa: E731
    nb, blk, mask = host(dm.slot_nb), host(dm.slot_blk), host(dm.slot_mask)
    nnz, idx, fps = host(dm.rows_nnz), host(dm.rows_idx), host(dm.fp_of_sp).reshape(3, dm.ns)
    bc, c = host(dm.slot_bc), mesh.n_cells // 2
    for pt in (0, 3, dm.ns - 1):
        reach = np.zeros((mesh.n_cells, dm.ns), dtype=bool)
        reach[c] = True
        for cell, slot in np.argwhere((nb == c).any(axis=2) & (bc == -1)):
            for fp in range(dm.nfp):
                src = (mask[cell, slot] >> fp) & 1
                row = blk[cell, slot, src] * dm.nfp + fp
                if nb[cell, slot, src] == c and pt in idx[row, :nnz[row]]:
                    reach[cell] |= fps[(0, 0, 1, 2)[slot]] == fp
        mut = torch.full(U.shape[:2], 1e-4, dtype=dt, device="cuda")
        mut[c, pt] = value
        R = host(dm.viscous_residual(U, mut, suppress=False))
        assert np.isfinite(R[..., 0]).all()
        assert np.array_equal(~np.isfinite(R[..., 1:]), np.repeat(reach[..., None], 4, axis=2)), pt
