"""GPU: per-case norms of a batch whose partial sums do not fit one group (4096 sums of 2048 values): a case
that takes them all, two that together exceed them, and more than 32 cases.  Bits of each case alone."""

import numpy as np
import pytest

from cases import freestream, wall_box

pytestmark = pytest.mark.gpu

BOXES = [(32, 32, 31), (2, 2, 3), (24, 24, 30), (24, 24, 30), (3, 3, 3)]


@pytest.mark.parametrize("order,boxes", [(2, BOXES), (1, [(2, 2, 3), (3, 3, 3)] * 17 + [(4, 4, 3)])])
def test_norms_past_one_group(order, boxes):
    import torch
    from autoflowcfd_amd.device import DeviceMesh, bc_params_table
    print(f"[gpu] norm partial sums P{order}, {len(boxes)} cases", flush=True)
    bcp = bc_params_table(freestream(0.15))
    mk = {n: DeviceMesh(wall_box(n, seed=1), order, dtype=torch.float32, bc_params=bcp) for n in set(boxes)}
    parts = [mk[n] for n in boxes]
    if order == 2:
        sums = [-(-q.n_cells * q.ns * 5 // 2048) for q in parts]
        assert sums[0] > 4096 and sums[2] + sums[3] > 4096
    batch = DeviceMesh.concat(parts, np.stack([bcp] * len(parts)), parts[0].ref_state)
    gen = torch.Generator(device="cuda").manual_seed(1)
    R = torch.randn((batch.n_cells, batch.ns, 5), generator=gen, device="cuda", dtype=torch.float32)
    out = torch.zeros(len(boxes), dtype=torch.float64, device="cuda")
    batch.residual_norm_cases(R, 5, out=out)
    first = 0
    for i, q in enumerate(parts):
        one = torch.zeros(1, dtype=torch.float64, device="cuda")
        q.residual_norm(R[first:first + q.n_cells].contiguous(), 5, out=one)
        first += q.n_cells
        assert float(one) == float(out[i]), i
