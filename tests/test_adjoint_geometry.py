"""evx_ch_rhs_vjp_workspace_bytes on the CPU (a query, no launch): extents of
which the adjoint refuses the launch, and extents beyond 32 bits, are answered
with a size and not with an arithmetic fault of the process."""
import ctypes as C
import subprocess
import sys

import pytest

from evoxels_amd import _lib

BIG = [(1, 4, 4, 1 << 32), (1, 4, 1 << 32, 4), (1, 1 << 32, 4, 4), (1 << 32, 4, 4, 4), (1, 1, 1, (1 << 31) + 64),
       (1, 1 << 20, 1 << 20, 1 << 20), (1, 3, (1 << 33) + 1, 1 << 33)]
PROG = """
import ctypes as C, sys
from evoxels_amd import _lib
g = _lib.EvxGrid()
g.channels, g.nx, g.ny, g.nz = (int(v) for v in sys.argv[1:])
n = C.c_size_t()
for dtype in (0, 1):
    st = _lib.load().evx_ch_rhs_vjp_workspace_bytes(dtype, C.byref(g), C.byref(n))
    assert st == 0 and n.value > 0, (st, n.value)
print("answered")
"""


@pytest.mark.parametrize("dims", BIG)
def test_query_answers_any_extent(dims):
    res = subprocess.run([sys.executable, "-c", PROG, *map(str, dims)], capture_output=True, text=True,
                         cwd=_lib.LIB_PATH.parents[1])
    assert res.returncode == 0 and "answered" in res.stdout, (res.returncode, res.stderr[-300:])


def test_sizes_of_ordinary_extents():
    for dtype in (0, 1):
        for dims in [(1, 1, 1, 1), (3, 5, 7, 11), (16, 128, 128, 128), (2, 4000, 3, 2)]:
            g = _lib.EvxGrid()
            g.channels, g.nx, g.ny, g.nz = dims
            n = C.c_size_t()
            assert _lib.load().evx_ch_rhs_vjp_workspace_bytes(dtype, C.byref(g), C.byref(n)) == 0
            assert n.value % 256 == 0 and n.value > 0


@pytest.mark.parametrize("dims", [(1, 4000, 12, 60), (1, 4000, 1, 60), (1, 65000, 2, 2)])
def test_long_thin_grids_fill_the_card(dims):
    """A block (with three partial sums) on each of 256 CUs, in place of a few
    blocks that march 60 planes and more one after another."""
    for dtype in (0, 1):
        g = _lib.EvxGrid()
        g.channels, g.nx, g.ny, g.nz = dims
        n = C.c_size_t()
        assert _lib.load().evx_ch_rhs_vjp_workspace_bytes(dtype, C.byref(g), C.byref(n)) == 0
        assert n.value >= 250 * 3 * 8  # equal chunks of whole planes: a few blocks fewer


def query(dtype, dims):
    g = _lib.EvxGrid()
    g.channels, g.nx, g.ny, g.nz = dims
    n = C.c_size_t()
    assert _lib.load().evx_ch_rhs_vjp_workspace_bytes(dtype, C.byref(g), C.byref(n)) == 0
    return n.value


@pytest.mark.parametrize("dims,separate", [
    ((1, 1, 1024, 1024), True), ((8, 2, 512, 512), True), ((16, 4000, 1, 4), True), ((4, 1024, 1, 1024), True),
    ((1, 1, 64, 64), False), ((1, 8, 8, 8), False), ((8, 100, 100, 100), False), ((16, 128, 128, 128), False),
    ((1, 3, 1 << 19, 4), False)])
def test_thin_grids_take_separate_kernels(dims, separate):
    """Where the streaming tiles would be mostly halo, mu, Gmu and the pointwise
    part are fields of the workspace; a grid of more block rows than a launch
    takes stays with the streaming kernel."""
    voxels = dims[0] * dims[1] * dims[2] * dims[3]
    for dtype, size in ((0, 4), (1, 8)):
        assert (query(dtype, dims) >= 3 * voxels * size) is separate
