"""GPU: the per-case norms of a batched mesh, whose launches take cases in groups (at most 32, and at most
4096 partial sums of 2048 values), have the bits of each case's norm alone; and the pseudo-step stage with
its filter at partly filled wavefronts, prisms and tets of one mesh, against the same sums in FP64 (1e-12;
FP32 2e-5: 64 products)."""

import numpy as np
import pytest

from cases import freestream, mixed_mesh, odd_prism_mesh, prim_to_cons, tet_box, wall_box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(1,), (3, 1, 2) * 11 + (1, 1), (2, 30, 30, 1)])
def test_norm_groups_have_the_bits_of_single_cases(sizes):
    import torch
    from autoflowcfd_amd.device import DeviceMesh, bc_params_table
    print(f"[gpu] norm groups of {len(sizes)} cases", flush=True)
    bcp = bc_params_table(freestream(0.15))
    mk = {n: DeviceMesh(wall_box((n, n, 3), seed=n), 1, dtype=torch.float32, bc_params=bcp) for n in set(sizes)}
    parts = [mk[n] for n in sizes]
    batch = DeviceMesh.concat(parts, np.stack([bcp] * len(parts)), parts[0].ref_state)
    gen = torch.Generator(device="cuda").manual_seed(1)
    R = torch.randn((batch.n_cells, 8, 5), generator=gen, device="cuda", dtype=torch.float32)
    out = torch.zeros(len(sizes), dtype=torch.float64, device="cuda")
    batch.residual_norm_cases(R, 5, out=out)
    first = 0
    for i, n in enumerate(sizes):
        one = torch.zeros(1, dtype=torch.float64, device="cuda")
        mk[n].residual_norm(R[first:first + mk[n].n_cells].contiguous(), 5, out=one)
        first += mk[n].n_cells
        assert float(one) == float(out[i]), i


@pytest.mark.parametrize("name,make", [("odd", odd_prism_mesh), ("mixed", mixed_mesh), ("tets", lambda: tet_box(2, seed=1))])
@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_stage_at_partly_filled_wavefronts(name, make, order, prec):
    import torch
    from autoflowcfd_amd.device import DeviceMesh, bc_params_table
    print(f"[gpu] rk stage {name} P{order} {prec}", flush=True)
    dt = torch.float64 if prec == "f64" else torch.float32
    Q0 = freestream(0.15)
    dm = DeviceMesh(make(), order, dtype=dt, bc_params=bc_params_table(Q0))
    rng = np.random.default_rng(2)
    shape = (dm.n_cells, dm.ns, 5)
    U = [torch.as_tensor(prim_to_cons(Q0) * (1 + 1e-2 * rng.uniform(-1, 1, shape)), dtype=dt, device="cuda") for _ in range(2)]
    R = torch.as_tensor(rng.uniform(-1, 1, shape), dtype=dt, device="cuda")
    step = torch.as_tensor(rng.uniform(0, 1e-3, shape[:2]), dtype=dt, device="cuda")
    out = torch.empty_like(R)
    dm.rk_stage(U[0], U[1], R, step, out, 0.75, 0.25, 0.25)
    V = 0.75 * U[0].double() + 0.25 * U[1].double() + 0.25 * step.double()[..., None] * R.double()
    n = dm.mesh.n_prism
    F = [f.double() for f in dm.filt]
    ref = torch.cat([F[0] @ V[:n], F[1] @ V[n:]])
    err = float((out.double() - ref).norm() / ref.norm())
    assert err < (1e-12 if prec == "f64" else 2e-5), err
