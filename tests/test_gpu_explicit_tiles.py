"""The explicit right-hand sides and steps at the edges of their tiles (16 x 64
points, float64 16 x 32 and, on grids of few rows, 8 x 64) next to every
ghost rule, against the oracle; and chunks of many planes, bitwise against
chunks of one plane."""
import warnings

import numpy as np
import pytest
import torch

import evoxels_amd as evx
from evoxels_amd.problem_definition import CoupledReactionDiffusion, ReactionDiffusion, TwoPhaseAllenCahn
from evoxels_amd.timesteppers import ForwardEuler, RungeKutta4
from evoxels_amd.voxelgrid import VoxelGridHip
from oracle import evoxels_oracle as O

pytestmark = pytest.mark.gpu

P, N = ("periodic", None), ("neumann", None)
D = ("dirichlet", (0.3, 0.8))
BCS = [(P, P, P), (N, D, P), (D, N, D), (P, D, D)]
# the arithmetic is the reference's, operation by operation
TOL = {"float32": 2e-6, "float64": 1e-14}


def problem(kind, shape, precision, bc, convention="cell_center"):
    vf = evx.VoxelFields(shape, tuple(s * n for s, n in zip((0.9, 1.1, 1.3), shape)), convention=convention)
    vf.precision = precision
    vg = VoxelGridHip(vf.grid_info(), precision=precision, device="cuda")
    og = O.OracleGrid(shape, vf.spacing, precision, convention)
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        if kind == "rd":
            return ReactionDiffusion(vg, D=0.7, bc=bc), lambda v: O.rd_rhs(v, og, bc, 0.7)
        if kind == "ac":
            return (TwoPhaseAllenCahn(vg, eps=2.5, gab=1.2, M=0.8, force=0.3, curvature=0.4, bc=bc),
                    lambda v: O.ac_rhs(v, og, bc, eps=2.5, gab=1.2, M=0.8, force=0.3, curvature=0.4))
        return (CoupledReactionDiffusion(vg, D_A=1.1, D_B=0.4, feed=0.05, kill=0.11),
                lambda v: O.coupled_rd_rhs(v, og, bc, 1.1, 0.4, 0.05, 0.11))


def state(kind, shape, precision):
    rng = np.random.default_rng(sum(shape))
    arr = 0.5 + 0.3 * rng.standard_normal(((2 if kind == "gs" else 1),) + shape)
    return torch.tensor(arr, dtype=getattr(torch, precision))


def check(kind, shape, precision, bc):
    p, rhs = problem(kind, shape, precision, bc)
    u = state(kind, shape, precision)
    ug = u.cuda()
    dt = 0.01
    k1 = rhs(u)
    k2 = rhs(u + 0.5 * dt * k1)
    k3 = rhs(u + 0.5 * dt * k2)
    k4 = rhs(u + dt * k3)
    for got, want in ((p.rhs(0.0, ug), k1), (ForwardEuler(p, dt).step(0.0, ug), u + dt * k1),
                      (RungeKutta4(p, dt).step(0.0, ug), u + (dt / 6) * (k1 + 2 * k2 + 2 * k3 + k4))):
        err = float((got.cpu() - want).abs().max() / want.abs().max())
        assert err < TOL[precision], (kind, shape, bc, err)


@pytest.mark.parametrize("precision", ["float32", "float64"])
@pytest.mark.parametrize("shape", [(3, 1, 33), (4, 8, 64), (3, 7, 65), (5, 9, 64), (2, 16, 64), (3, 24, 128), (2, 32, 32),
                                   (3, 17, 40), (1, 40, 63), (6, 41, 66), (2, 8, 32)])
def test_tile_edges(shape, precision):
    for kind in ("rd", "ac", "gs"):
        for bc in BCS if kind != "gs" else [(P, P, P)]:
            check(kind, shape, precision, bc)


# A grid that fits one resident round has chunks of one plane (checked against
# the oracle above), so the slots and registers that a chunk hands on from plane
# to plane take part only in copies of the field that fill the card several
# times: channels with any walls, or periods of y and z.  A copy's values do
# not depend on its neighbours, so each equals the small result bit for bit.
@pytest.mark.parametrize("precision", ["float32", "float64"])
@pytest.mark.parametrize("planes", [2, 3, 4, 5, 6, 7, 11])
@pytest.mark.parametrize("kind,bc,convention", [
    ("rd", (D, D, D), "cell_center"), ("rd", (N, D, P), "cell_center"), ("rd", (D, P, P), "staggered_x"),
    ("rd", (N, P, P), "staggered_x"), ("ac", (D, N, D), "cell_center"), ("ac", (P, D, N), "cell_center"),
    ("ac", (N, P, P), "staggered_x"), ("ac", (D, P, P), "staggered_x"), ("gs", (P, P, P), "cell_center")])
def test_long_chunks_equal_chunks_of_one_plane(kind, bc, convention, planes, precision):
    inner = (planes, 16, 64) if kind == "gs" else (planes, 17 if planes % 2 else 16, 40)  # float64: both tiles
    nodes = (planes + (2 if convention == "staggered_x" else 0),) + inner[1:]
    small, _ = problem(kind, nodes, precision, bc, convention)
    u = state(kind, inner, precision).cuda()
    if kind == "gs":
        big, _ = problem(kind, (planes, 16 * 64, 64 * 80), precision, bc)
        big.vg.div_dx_host, big.vg.div_dx2_host = small.vg.div_dx_host, small.vg.div_dx2_host
        copies = (1, 1, 64, 80)
    else:
        big, copies = small, (4096, 1, 1, 1)
    dt = 0.01
    for step in (lambda p, v: p.rhs(0.0, v), lambda p, v: ForwardEuler(p, dt).step(0.0, v),
                 lambda p, v: RungeKutta4(p, dt).step(0.0, v)):
        assert torch.equal(step(big, u.repeat(copies)), step(small, u).repeat(copies))
