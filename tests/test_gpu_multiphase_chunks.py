"""The one-launch multiphase right-hand side in chunks that reuse the slots of its
ring of four planes: three to eleven planes a chunk, bitwise against chunks of
one plane (which the other multiphase tests hold against the oracle)."""
import numpy as np
import pytest
import torch

import evoxels_amd as evx
from evoxels_amd.problem_definition import MultiPhaseAllenCahn
from evoxels_amd.timesteppers import ForwardEuler, RungeKutta4
from evoxels_amd.voxelgrid import VoxelGridHip

pytestmark = pytest.mark.gpu

COPIES = (40, 64)  # tiles of 16 x 32 points along y and z: more than a resident round


def problem(shape, precision, bc, convention, **kw):
    vf = evx.VoxelFields(shape, tuple(float(n) for n in shape), convention=convention)
    vf.precision = precision
    return MultiPhaseAllenCahn(VoxelGridHip(vf.grid_info(), precision=precision, device="cuda"), eps=2.5, bc=bc, **kw)


# A field that repeats along periodic y and z: every copy sees the same
# neighbours, and a grid of one tile runs in chunks of one plane.
@pytest.mark.parametrize("precision", ["float32", "float64"])
@pytest.mark.parametrize("planes", [1, 2, 3, 4, 5, 6, 8, 11])
@pytest.mark.parametrize("n,fast,curvature,wall,convention", [
    (3, True, 1.0, "periodic", "cell_center"), (3, True, 1.0, "neumann", "cell_center"),
    (2, False, 1.0, ("dirichlet", (0.3, 0.8)), "cell_center"), (4, True, 0.5, "neumann", "cell_center"),
    (6, False, 0.5, "periodic", "cell_center"), (3, True, 1.0, ("dirichlet", (0.3, 0.8)), "staggered_x"),
    (2, False, 0.5, "neumann", "staggered_x")])
@pytest.mark.filterwarnings("ignore:Applying Dirichlet")
def test_long_chunks_equal_chunks_of_one_plane(n, fast, curvature, wall, convention, planes, precision):
    if wall == "neumann" and convention == "staggered_x" and planes < 2:
        pytest.skip("the staggered zero-flux rule needs two interior planes")
    nx = planes + (2 if convention == "staggered_x" else 0)
    bc = (wall, "periodic", "periodic")
    kw = dict(fast=fast, curvature=curvature)
    small = problem((nx, 16, 32), precision, bc, convention, **kw)
    big = problem((nx, 16 * COPIES[0], 32 * COPIES[1]), precision, bc, convention, **kw)
    assert big.vg.div_dx_host == small.vg.div_dx_host
    rng = np.random.default_rng(planes + n)
    arr = 0.02 + rng.dirichlet([1.5] * n, size=(planes, 16, 32)).transpose(3, 0, 1, 2)
    u = torch.tensor(arr, dtype=small.vg.precision, device="cuda")
    v = u.repeat(1, 1, *COPIES)
    assert small.fused_for(u) and big.fused_for(v)
    for step in (lambda p, w: p.rhs(0.0, w), lambda p, w: ForwardEuler(p, 0.05).step(0.0, w),
                 lambda p, w: RungeKutta4(p, 0.05).step(0.0, w)):
        assert torch.equal(step(big, v), step(small, u).repeat(1, 1, *COPIES))
