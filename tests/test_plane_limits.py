"""Planes of more points than a kernel's 32-bit in-plane offsets reach are
refused before any launch (CPU: the pointers are never followed)."""
import ctypes as C

import pytest

from evoxels_amd import _lib

PER = (("periodic", None),) * 3


def calls(lib, grid, dtype):
    b, e = _lib.make_bc(PER), _lib.make_epilogue()
    a = (dtype, C.c_void_p(256), C.c_void_p(512), C.byref(grid), C.byref(b))
    return {"rd": lambda: lib.evx_rd_rhs(*a, 1.0, C.byref(e), None),
            "ch": lambda: lib.evx_ch_rhs(*a, 3.0, 1.0, C.byref(e), None),
            "ac": lambda: lib.evx_ac_rhs(*a, 2.0, 1.0, 1.0, 0.0, 1.0, C.byref(e), None),
            "gs": lambda: lib.evx_coupled_rd_rhs(*a, 1.0, 0.5, 0.05, 0.1, C.byref(e), None),
            "mp": lambda: lib.evx_multiphase_ac_rhs(*a, 2.0, 1.0, 1.0, 1.0, 0, C.byref(e), None)}


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("kind", ["rd", "ch", "ac", "gs", "mp"])
@pytest.mark.parametrize("ny,nz", [(65536, 65536), (1, 1 << 32), (1 << 33, 3), (1 << 62, 1 << 62)])
def test_wide_planes_are_refused(kind, dtype, ny, nz):
    lib = _lib.load()
    g = _lib.make_grid((2 if kind == "gs" else 1, 1, ny, nz), (1, 1, 1), (1, 1, 1))
    assert calls(lib, g, dtype)[kind]() == _lib.EVX_ERR_UNSUPPORTED
    assert "plane" in _lib.last_error()
