"""GPU: the outlier zeroing of the SST transport where FP64 rates lie beyond the FP32 range (k of 1e60, a
diverging solve): the decisions are those of the FP64 rule, the oracle's.  Tolerance 1e-9 of the largest
increment, which the cells of varying k set; an entry zeroed on one side only is of that size."""

import numpy as np
import pytest

from cases import freestream, prim_to_cons, wall_box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [1, 2])
def test_zeroing_beyond_the_fp32_range(order):
    import torch
    from autoflowcfd_amd.device import DeviceMesh, bc_params_table
    from autoflowcfd_amd.mesh import BC_WALL
    from oracle import fr_ops, sst
    from oracle.faces import build_flat_faces
    from oracle.geometry import Geometry
    from oracle.time_step import local_time_step, update_primitives
    print(f"[gpu] sst zeroing beyond the FP32 range P{order}", flush=True)
    mesh = wall_box(seed=2)
    ops = fr_ops.generate_operators(order)
    g = Geometry(mesh, ops)
    fl = build_flat_faces(mesh, ops)
    Q0 = freestream(0.15)
    U = np.broadcast_to(prim_to_cons(Q0), (mesh.n_cells, ops.n_sps, 5)).copy()
    rng = np.random.default_rng(0)
    k, w = np.full((mesh.n_cells, ops.n_sps), 1e60), np.full((mesh.n_cells, ops.n_sps), 2660.0)
    c = rng.permutation(mesh.n_cells)
    for i in c[:4]:
        k[i, rng.integers(ops.n_sps)] *= 1.5
    k[c[4:8]] *= 1.0 + 0.2 * rng.uniform(-1, 1, (4, ops.n_sps))
    mu, hit = 1.8e-5, []
    orig = sst.suppress_outliers

    def watched(R, Uref, *a, **kw):
        out = orig(R, Uref, *a, **kw)
        zeroed = ((out == 0) & (R != 0)).reshape(mesh.n_cells, -1).any(axis=1)
        beyond = (np.abs(R).reshape(mesh.n_cells, -1) > np.finfo(np.float32).max).sum(axis=1) > ops.n_sps // 2
        hit.append(int((zeroed & beyond).sum()))
        return out
    sst.suppress_outliers = watched
    try:
        d = sst.wall_distance(g.sps_xyz, mesh.nodes[mesh.wall_nodes])
        dtl = local_time_step(update_primitives(U), g, order, mu, None)
        kn, wn, _, _, _ = sst.turbulence_step(U, k, w, g, ops, fl, d, dtl, mu, fl.bc == BC_WALL)
    finally:
        sst.suppress_outliers = orig
    assert hit[0] > 0, "no cell that is zeroed has its median beyond the FP32 range"
    dm = DeviceMesh(mesh, order, dtype=torch.float64, bc_params=bc_params_table(Q0), turbulence="SST")
    Ud, kd, wd = (torch.as_tensor(x, dtype=torch.float64, device="cuda").contiguous() for x in (U, k, w))
    dtd = dm.local_time_step(Ud, mu=mu)
    dm.sst_step(Ud, kd, wd, dtd, torch.zeros_like(kd), torch.zeros_like(kd), mu=mu)
    err = np.abs(kd.cpu().numpy() - kn).max() / np.abs(kn - k).max()
    assert err < 1e-9, f"k {err:.3e}"
