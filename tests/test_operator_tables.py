"""The residual and SST entry points refuse a mesh description without an operator table that their kernels
read for a cell type present, before any GPU call; tables of an absent type are not asked for."""

import ctypes

import pytest

CALLS = {
    "inviscid": lambda lib, m, x: lib.afr_inviscid_residual(m, x, x, 1, None),
    "primitives": lambda lib, m, x: lib.afr_inviscid_from_primitives(m, x, x, x, 1, None),
    "viscous": lambda lib, m, x: lib.afr_viscous_residual(m, x, None, x, 1.8e-5, 0.72, 0.9, 1, None),
    "volume": lambda lib, m, x: lib.afr_viscous_volume(m, x, None, 1.8e-5, 0.72, 0.9, None),
    "full": lambda lib, m, x: lib.afr_residual(m, x, None, x, 1.8e-5, 0.72, 0.9, 1, None),
    "sst": lambda lib, m, x: lib.afr_sst_step(m, x, x, x, x, x, x, x, None, 1.8e-5, None),
}
# table -> calls whose kernels read it (op and c2f: tets only)
READS = {"E": CALLS, "D": ("viscous", "volume", "full", "sst"), "op": ("inviscid", "primitives", "full"),
         "c2f": ("inviscid", "primitives", "full")}


@pytest.mark.parametrize("kind,table,call", [(k, t, c) for k in ("prism", "tet") for t in sorted(READS)
                                             for c in sorted(READS[t]) if k == "tet" or t in ("E", "D")])
def test_missing_operator_is_an_error(kind, table, call):
    from autoflowcfd_amd import _lib
    ct = 0 if kind == "prism" else 1
    lib = _lib.load()
    d = _lib.AfrMeshDesc()
    for name, typ in d._fields_:           # every pointer set (none is followed before the check), as a caller would
        if typ is _lib.c_vp:
            setattr(d, name, 4096)
        elif typ is _lib.c_vp * 2:
            setattr(d, name, typ(4096, 4096))
    d.cell_case = d.state_ref = None
    d.abi_version, d.order, d.dtype, d.n_rows, d.rows_knz = _lib.ABI_VERSION, 1, 0, 4, 4
    d.n_cells, d.n_prism, d.n_records = 3, 3 if ct == 0 else 0, 1
    for name in ("E", "D", "op", "c2f"):   # of the type that is not there: nothing
        getattr(d, name)[1 - ct] = None
    getattr(d, table)[ct] = None
    m = ctypes.c_void_p()
    _lib.check(lib.afr_mesh_create(ctypes.byref(d), ctypes.byref(m)), "afr_mesh_create")
    try:
        with pytest.raises(RuntimeError, match="no operator tables|no viscous work buffers"):
            _lib.check(CALLS[call](lib, m, ctypes.c_void_p(4096)), call)
    finally:
        lib.afr_mesh_destroy(m)
