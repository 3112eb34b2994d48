"""GPU: the mean-flow residual takes the width of an interpolation row from the row tables; the hint bit of
the slot masks (bit 30) changes nothing."""

import pytest

from cases import freestream, mixed_mesh, rotated_prism_box, wall_box
from cases import smooth_state

pytestmark = pytest.mark.gpu

MESHES = {"wallbox": lambda: wall_box(seed=4), "rotated": lambda: rotated_prism_box(seed=2), "mixed": mixed_mesh}


def _device(mesh, order, dtype):
    import numpy as np
    import torch
    from autoflowcfd_amd.device import DeviceMesh, bc_params_table
    from autoflowcfd_amd.geometry import map_ref
    Q0 = freestream(0.15, 4.0)
    dm = DeviceMesh(mesh, order, dtype=dtype, bc_params=bc_params_table(Q0))
    xyz = np.zeros((mesh.n_cells, dm.ns, 3))
    if mesh.n_prism:
        xyz[:mesh.n_prism] = map_ref(True, dm.T.sps, mesh.nodes[mesh.prism_conn])
    if mesh.n_tet:
        xyz[mesh.n_prism:] = map_ref(False, dm.T.sps, mesh.nodes[mesh.tet_conn])
    U = torch.as_tensor(smooth_state(xyz, Q0, amp=2e-2, seed=3), dtype=dtype, device="cuda").contiguous()
    mut = torch.full(U.shape[:2], 1e-4, dtype=dtype, device="cuda")
    return dm, U, mut


def _residuals(dm, U, mut):
    return [dm.residual(U, mut), dm.inviscid_residual(U), dm.viscous_residual(U, mut)]


@pytest.mark.parametrize("name", sorted(MESHES))
@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("prec", ["f32", "f64"])
def test_wide_row_hint_changes_nothing(name, order, prec):
    import torch
    print(f"[gpu] wide-row hint {name} P{order} {prec}", flush=True)
    dm, U, mut = _device(MESHES[name](), order, torch.float32 if prec == "f32" else torch.float64)
    assert int(dm.rows_nnz.max()) > order + 1
    ref = _residuals(dm, U, mut)
    mask = dm.slot_mask.clone()
    for bits in (mask & ~(1 << 30), mask | 1 << 30):
        dm.slot_mask.copy_(bits)
        for a, b in zip(_residuals(dm, U, mut), ref):
            assert torch.equal(a, b)
