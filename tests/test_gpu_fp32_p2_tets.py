"""GPU: the FP32 kernels on P2 tets (alone and beside prisms; partly filled tiles of 12 cells, waves of 2)
against the FP64 kernels on the same FP32-rounded state: the inviscid residual without outlier zeroing (the
medians of cancelling sums are round-off) and the SST step.

Tolerances: n u sum |a||b| for the sums of n products that the volume terms form (u = 2^-24; inviscid 27 + 81
terms, SST 27 + 9 + 3, once for the gradient and once for the divergence), from the mesh's own operators
(derivative rows of up to 9e3, restricted divergence up to 3e6) and fields, in the norm of the comparison.
SST: increments hold products of two gradients and a divergence, hence twice the gradients' relative bound
and once the divergence's, of the largest increment."""

import numpy as np
import pytest

from cases import freestream, mixed_mesh, smooth_state, tet_box

pytestmark = pytest.mark.gpu

U24, MU = 2.0 ** -24, 1.8e-5
NAMES = ["tet1", "tet2", "tet7", "tet8", "tet12", "tet13", "box", "mixed"]


def _mesh(name):
    from autoflowcfd_amd.mesh import BC_FARFIELD, BC_WALL, mesh_from_cells
    if name == "mixed":
        m = mixed_mesh()
    elif name == "box":
        m = tet_box(3, seed=1)
    else:
        src = tet_box(2, seed=1)
        m = mesh_from_cells(src.nodes, None, src.tet_conn[:int(name[3:])], default_bc=BC_FARFIELD)
    fr = m.faces
    low = np.flatnonzero(fr.is_boundary)[:3]
    fr.bc[low] = BC_WALL
    m.wall_nodes = np.unique(fr.node_ids[low])
    m.wall_nodes = m.wall_nodes[m.wall_nodes >= 0]
    return m


def _parts(mesh, T):
    from autoflowcfd_amd.geometry import cell_block_metrics
    geo = cell_block_metrics(mesh, T, dtype=np.float64)
    for ct, sl in ((0, slice(0, mesh.n_prism)), (1, slice(mesh.n_prism, mesh.n_cells))):
        if sl.stop > sl.start:
            yield sl, np.transpose(T.D[ct], (2, 0, 1)), T.c2f[ct], T.Op[ct], *(geo[k][sl] for k in ("det", "adj", "adj_fine"))


def _inviscid_bound(mesh, T, U, Q0):
    """Round-off bound of the inviscid volume term, every entry."""
    Q = np.empty_like(U)
    Q[..., 0], Q[..., 1:4] = U[..., 0], U[..., 1:4] / U[..., :1]
    Q[..., 4] = 0.4 * (U[..., 4] - 0.5 * Q[..., 0] * (Q[..., 1:4] ** 2).sum(-1))
    inv = np.zeros_like(U)
    r0, vm, p0 = Q0[0], np.abs(Q0[1:4]), Q0[4]
    H = 3.5 * p0 / r0 + 0.5 * (vm ** 2).sum()
    for sl, _, c2f, Op, det, _, adjf in _parts(mesh, T):
        qf = np.abs(c2f) @ np.abs(Q[sl] - Q0)
        dr, dv, dp = qf[..., 0], qf[..., 1:4], qf[..., 4]
        dF = np.zeros(qf.shape[:2] + (3, 5))             # sizes of F(Q0 + dq) - F(Q0)
        for i in range(3):
            dm = r0 * dv[..., i] + dr * vm[i]
            dF[..., i, 0] = dm
            dF[..., i, 1:4] = vm * dm[..., None] + r0 * vm[i] * dv
            dF[..., i, 1 + i] += dp
            dF[..., i, 4] = H * dm + r0 * vm[i] * (3.5 * (dp / r0 + p0 * dr / r0 ** 2) + (vm * dv).sum(-1))
        Ft = np.einsum("cjmi,cjiv->cmjv", np.abs(adjf), dF)
        inv[sl] = 108 * U24 * np.einsum("smj,cmjv->csv", np.abs(Op).reshape(T.ns, 3, -1), Ft) / det[..., None]
    return inv


def _sst_bound(mesh, T, U, k, w):
    grad, div = 0.0, 0.0
    for sl, D, _, _, det, adj, _ in _parts(mesh, T):
        for x in (U[sl, :, 1:4], k[sl, :, None], w[sl, :, None]):
            x = x - x[:, :1]
            g = np.einsum("csmn,cmsf->csnf", adj, np.einsum("mst,ctf->cmsf", D, x)) / det[..., None, None]
            ga = np.einsum("csmn,cmsf->csnf", np.abs(adj), np.einsum("mst,ctf->cmsf", np.abs(D), np.abs(x))) / det[..., None, None]
            grad = max(grad, 39 * U24 * ga.max() / np.abs(g).max())
        for phi in (k, w):
            F = np.einsum("csmn,csn->csm", adj, U[sl, :, 1:4]) * phi[sl, :, None]
            F = F - F[:, :1]
            size = (np.einsum("mst,ctm->cs", np.abs(D), np.abs(F)) / det).max()
            div = max(div, 39 * U24 * size / np.abs(np.einsum("mst,ctm->cs", D, F) / det).max())
    return 2 * grad + div


@pytest.mark.parametrize("name", NAMES)
def test_fp32_p2_tets_match_fp64(name):
    import torch
    from autoflowcfd_amd.device import DeviceMesh, bc_params_table
    from autoflowcfd_amd.fr_tables import tables
    from autoflowcfd_amd.geometry import map_ref
    print(f"[gpu] FP32 P2 tets {name}", flush=True)
    mesh, T, Q0 = _mesh(name), tables(2), freestream(0.15, 4.0)
    xyz = np.zeros((mesh.n_cells, T.ns, 3))
    if mesh.n_prism:
        xyz[:mesh.n_prism] = map_ref(True, T.sps, mesh.nodes[mesh.prism_conn])
    xyz[mesh.n_prism:] = map_ref(False, T.sps, mesh.nodes[mesh.tet_conn])
    rng = np.random.default_rng(4)
    f32 = lambda x: x.astype(np.float32).astype(np.float64)  # noqa: E731
    U = f32(smooth_state(xyz, Q0, seed=3))
    k, w = (f32(x * (1.0 + 0.2 * rng.uniform(-1, 1, U.shape[:2]))) for x in (0.39, 2660.0))
    out = {}
    for dt in (torch.float32, torch.float64):
        dm = DeviceMesh(mesh, 2, dtype=dt, bc_params=bc_params_table(Q0), turbulence="SST")
        Ud, kd, wd = (torch.as_tensor(x, dtype=dt, device="cuda").contiguous() for x in (U, k, w))
        R = dm.inviscid_residual(Ud, suppress=False)
        dtl = torch.full(U.shape[:2], 1e-6, dtype=dt, device="cuda")
        nut, mt = torch.zeros_like(kd), torch.zeros_like(kd)
        dm.sst_step(Ud, kd, wd, dtl, nut, mt, mu=MU)
        out[dt] = [x.double().cpu().numpy() for x in (R, kd, wd, nut)]
    a, b = out[torch.float32], out[torch.float64]
    bound = _inviscid_bound(mesh, T, U, Q0)
    for v in range(5):
        err, lim = (float(np.linalg.norm(x)) for x in (a[0][..., v] - b[0][..., v], bound[..., v]))
        assert err <= lim, f"inviscid {v}: {err:.3e} > {lim:.3e}"
    tol = _sst_bound(mesh, T, U, k, w)
    assert tol < 0.1
    for x, y, x0 in ((a[1], b[1], k), (a[2], b[2], w)):
        # (storing the field in FP32 rounds the increment by its own unit)
        assert np.abs(x - y).max() <= tol * np.abs(y - x0).max() + U24 * np.abs(y).max()
    assert np.abs(a[3] - b[3]).max() <= tol * np.abs(b[3]).max()
