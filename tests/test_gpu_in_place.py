"""GPU: a residual written over its own state, or over a part of it, has the bits of one written elsewhere.
The spiked state sends columns to the outlier rule's median, which also reads mean |U|."""

import numpy as np
import pytest

from cases import freestream, mixed_mesh, prim_to_cons, tet_box, wall_box

pytestmark = pytest.mark.gpu

MESHES = {"prism": lambda: wall_box(seed=1), "tet": lambda: tet_box(2, seed=1), "mixed": mixed_mesh}


@pytest.mark.parametrize("name,order,prec", [(n, o, p) for n in sorted(MESHES) for o in (1, 2) for p in ("f32", "f64")]
                         + [("tet", 3, "f64")])
def test_residual_over_its_state(name, order, prec):
    import torch
    from autoflowcfd_amd.device import DeviceMesh, bc_params_table
    print(f"[gpu] residual in place {name} P{order} {prec}", flush=True)
    dt = torch.float32 if prec == "f32" else torch.float64
    mesh = MESHES[name]()
    Q0 = freestream(0.2, 3.0)
    dm = DeviceMesh(mesh, order, dtype=dt, bc_params=bc_params_table(Q0))
    rng = np.random.default_rng(0)
    U = np.broadcast_to(prim_to_cons(Q0), (mesh.n_cells, dm.ns, 5)).copy()
    for c in range(0, mesh.n_cells, 3):
        U[c, rng.integers(dm.ns)] *= 1.01
    Ud = torch.as_tensor(U, dtype=dt, device="cuda").contiguous()
    calls = {"full": lambda X, R: dm.residual(X, None, R), "inviscid": dm.inviscid_residual,
             "viscous": lambda X, R: dm.viscous_residual(X, None, R)}
    n = Ud.numel()
    for what, call in calls.items():
        ref = call(Ud, torch.empty_like(Ud)).clone()
        for shift in (0, dm.ns * 5, -7):                 # in place, a cell further on, some values before
            buf = torch.empty(n + 2 * abs(shift), dtype=dt, device="cuda")
            X = buf[abs(shift):abs(shift) + n].view_as(Ud)
            R = buf[abs(shift) + shift:abs(shift) + shift + n].view_as(Ud)
            X.copy_(Ud)
            assert torch.equal(call(X, R), ref), (what, shift)
