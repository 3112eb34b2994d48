"""GPU: the mean-flow volume and interface kernels at the edges of their cell tiles, against the FP64
oracle, and their 64-bit index form against the 32-bit one.

Tolerances (relative L2): FP64 1e-10, P2 tets 1e-7 (collapsed derivative operators up to 4e5); FP32
1e-5 on the FP32-rounded state.
"""

import numpy as np
import pytest

from cases import freestream, prim_to_cons, smooth_state, tet_box, wall_box

pytestmark = pytest.mark.gpu

MU = 1.8e-5
# interface tiles: 12 / 5 prisms (P1 / P2), 16 / 7 tets; volume tiles: 4 / 3 prisms,
# 16 (FP64) or 12 tets; gradient passes: 8 cells (P1) or 2 (P2) per wavefront.  Two P2 tets have more row
# fragments than scratch and take the FP64 interface kernel without matrix products, 13 take the other
EDGES = ([("prism", 1, n) for n in (1, 8, 11, 12, 13)] + [("prism", 2, n) for n in (1, 4, 5, 6, 7)]
         + [("tet", 1, n) for n in (1, 12, 16, 17)] + [("tet", 2, n) for n in (1, 2, 7, 8, 13)])


@pytest.mark.parametrize("kind,order,n", EDGES)
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_tile_edges_match_oracle(kind, order, n, prec):
    import torch
    from autoflowcfd_amd.device import DeviceMesh, bc_params_table
    from autoflowcfd_amd.mesh import BC_FARFIELD, mesh_from_cells
    from oracle import fr_ops
    from oracle.faces import build_flat_faces
    from oracle.geometry import Geometry
    from oracle.residual import inviscid_residual, viscous_residual
    if prec == "f32" and kind == "tet" and order > 1:
        pytest.skip("tets above P1 are computed in FP64")
    print(f"[gpu] tile edges {kind} P{order} n={n} {prec}", flush=True)
    src = wall_box((3, 2, 2), seed=2) if kind == "prism" else tet_box(2, seed=1)
    mesh = (mesh_from_cells(src.nodes, src.prism_conn[:n], default_bc=BC_FARFIELD) if kind == "prism"
            else mesh_from_cells(src.nodes, None, src.tet_conn[:n], default_bc=BC_FARFIELD))
    Q0 = freestream(0.15)
    bcp = bc_params_table(Q0)
    bcd = {c: bcp[c] for c in range(8)}
    ops = fr_ops.generate_operators(order)
    g = Geometry(mesh, ops)
    fl = build_flat_faces(mesh, ops)
    U = smooth_state(g.sps_xyz, Q0, seed=3)
    mut = MU * np.random.default_rng(4).uniform(0.0, 50.0, size=U.shape[:2])
    dt = torch.float64 if prec == "f64" else torch.float32
    if prec == "f32":
        U, mut = U.astype(np.float32).astype(np.float64), mut.astype(np.float32).astype(np.float64)
    Ri = inviscid_residual(U, g, ops, fl, bcd)
    Rv = viscous_residual(U, g, ops, fl, bcd, MU, mu_t=mut)
    dm = DeviceMesh(mesh, order, dtype=dt, bc_params=bcp)
    Ud = torch.as_tensor(U, dtype=dt, device="cuda").contiguous()
    md = torch.as_tensor(mut, dtype=dt, device="cuda").contiguous()
    tol = 1e-5 if prec == "f32" else {("tet", 2): 1e-7}.get((kind, order), 1e-10)
    for name, dev, ref in (("inviscid", dm.inviscid_residual(Ud), Ri), ("viscous", dm.viscous_residual(Ud, md, mu=MU), Rv),
                           ("full", dm.residual(Ud, md, mu=MU), Ri + Rv)):
        err = np.linalg.norm(dev.double().cpu().numpy() - ref) / np.linalg.norm(ref)
        assert err < tol, f"{name} {kind} P{order} n={n}: rel L2 {err:.3e}"


def test_offsets_past_4_gib_match_small_mesh():
    """546,750 P3 tets (an 4.2 GiB pack: the 64-bit index form) with a disturbed 5^3-hex corner, against
    the same corner as a mesh of its own: cells away from the cut must agree.  Spacings are powers of
    two; the translated geometry still rounds at 1e-16 x 45 spacings, times operators of ~1e6: 1e-6."""
    import torch
    from autoflowcfd_amd.device import DeviceMesh, bc_params_table
    from autoflowcfd_amd.mesh import hex_box, mesh_from_cells
    N, m, h = 45, 5, 1.0 / 64
    print("[gpu] 64-bit offsets", flush=True)
    big = hex_box(N, N, N, N * h, N * h, N * h, split="tet", permute=False, topology="gpu")
    i = np.arange(N) >= N - m
    corner = np.repeat((i[:, None, None] & i[None, :, None] & i[None, None, :]).ravel(), 6)
    inner = np.arange(N) >= N - m + 1
    keep = np.repeat((inner[:, None, None] & inner[None, :, None] & inner[None, None, :]).ravel(), 6)[corner]
    from autoflowcfd_amd.mesh import BC_FARFIELD
    small = mesh_from_cells(big.nodes, None, big.tet_conn[corner], default_bc=BC_FARFIELD, topology="gpu")
    assert np.array_equal(small.tet_conn, big.tet_conn[corner])
    Q0 = freestream(0.15)
    rng = np.random.default_rng(5)
    Q = Q0 * (1.0 + 1e-2 * rng.uniform(-1, 1, (small.n_cells, 64, 5)))
    sub = torch.as_tensor(prim_to_cons(Q), device="cuda")
    out = []
    for mesh, sel in ((small, None), (big, torch.as_tensor(np.flatnonzero(corner), device="cuda"))):
        dm = DeviceMesh(mesh, 3, dtype=torch.float64, bc_params=bc_params_table(Q0), metrics="gpu")
        U = sub
        if sel is not None:
            U = torch.as_tensor(prim_to_cons(Q0), device="cuda").expand(mesh.n_cells, 64, 5).contiguous()
            U[sel] = sub
        R = torch.stack([dm.residual(U, None, mu=MU, suppress=False), dm.inviscid_residual(U, suppress=False)])
        out.append((R if sel is None else R[:, sel])[:, torch.as_tensor(keep, device="cuda")].cpu().numpy())
        del dm, U, R
        torch.cuda.empty_cache()
    err = np.linalg.norm(out[1] - out[0]) / np.linalg.norm(out[0])
    assert err < 1e-6, f"rel L2 {err:.3e}"
