"""The autotuner against a stub mesh (no GPU): every grid size is timed once per kernel, a choice cached for
other kernels (a key without their revision) or other cell types is not taken, and a cached one of its own is."""

import json
from types import SimpleNamespace

import pytest


class _Lib:
    def __init__(self):
        self.grid, self.variant = {}, {}

    def afr_mesh_set_grid(self, handle, kernel, cap):
        self.grid[kernel] = cap
        return 0

    def afr_mesh_set_variant(self, handle, kernel, variant):
        self.variant[kernel] = variant
        return 0


def _mesh(n_prism, n_tet):
    import torch
    call = lambda *a, **k: None  # noqa: E731
    return SimpleNamespace(n_cells=n_prism + n_tet, n_prism=n_prism, ns=8, order=1, dtype=torch.float32, device="cpu", handle=None,
                           lib=_Lib(), turbulence=None, mesh=SimpleNamespace(n_prism=n_prism, n_tet=n_tet),
                           work_q=None, work_umean=None, viscous_volume=call, residual=call,
                           inviscid_from_primitives=call)


@pytest.fixture
def tuner(monkeypatch):
    import torch
    from autoflowcfd_amd import autotune as at
    timed = []

    def clock(fn, reps):
        fn()
        timed.append(fn)
        return {16: 1.0}.get(at._stub.lib.grid[max(at._stub.lib.grid)], 2.0)
    monkeypatch.setattr(torch.cuda, "get_device_name", lambda *a: "stub")
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: None)
    monkeypatch.setattr(at, "_time", clock)
    monkeypatch.setattr(at, "_memo", {})

    def run(dm, **kw):
        at._stub = dm
        timed.clear()
        return at.autotune(dm, torch.zeros(2, 8, 5), candidates=(0, 16, 64), **kw), len(timed)
    yield run
    del at._stub


def test_each_grid_is_timed_once(tuner):
    out, n = tuner(_mesh(100, 0))
    assert set(out) == {"prism_inviscid", "visc_volume", "visc_iface"} and n == 3 * 3
    assert all(v["variant"] == 0 for v in out.values())


def test_cached_choices_of_other_kernels_or_cells_are_not_taken(tuner, tmp_path):
    path = tmp_path / "cache.json"
    path.write_text(json.dumps({f"stub|P1|float32|{k}|2^7": {"grid": 64, "variant": 1}
                                for k in ("prism_inviscid", "visc_volume", "visc_iface")}))
    out, n = tuner(_mesh(100, 0), cache_path=str(path))
    assert n == 9 and out["visc_iface"]["grid"] == 16
    assert tuner(_mesh(100, 0), cache_path=str(path))[1] == 0           # its own choice: reused
    assert tuner(_mesh(0, 100), cache_path=str(path))[1] == 9           # tets of the same count: timed
    assert tuner(_mesh(50, 50), cache_path=str(path))[1] == 12
