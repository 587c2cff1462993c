"""The one-launch multiphase Allen-Cahn right-hand side: one to eight phases,
tile edges in y and z, x chunks shorter and longer than the plane ring, every
ghost rule (staggered_x included), against the oracle; its Euler and RK4
epilogues bitwise against the same composition of right-hand sides."""
import warnings

import numpy as np
import pytest
import torch

import evoxels_amd as evx
from evoxels_amd.problem_definition import MultiPhaseAllenCahn
from evoxels_amd.timesteppers import ForwardEuler, RungeKutta4
from evoxels_amd.voxelgrid import VoxelGridHip
from oracle import evoxels_oracle as O

pytestmark = pytest.mark.gpu

P, N = ("periodic", None), ("neumann", None)
D = ("dirichlet", (0.3, 0.8))
TOL = {"float32": 4e-6, "float64": 1e-12}  # the reference's operations in its order: a few roundings


def build(shape, precision, bc, convention="cell_center", **kw):
    vf = evx.VoxelFields(shape, tuple(s * n for s, n in zip((0.9, 1.1, 1.3), shape)), convention=convention)
    vf.precision = precision
    vg = VoxelGridHip(vf.grid_info(), precision=precision, device="cuda")
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        return MultiPhaseAllenCahn(vg, eps=2.5, gab=1.2, M=0.8, bc=bc, **kw), O.OracleGrid(shape, vf.spacing, precision,
                                                                                           convention)


def phases(shape, n, seed):
    rng = np.random.default_rng(seed)
    a = rng.dirichlet([1.5] * n, size=shape).transpose(3, 0, 1, 2) + 0.08 * rng.standard_normal((n,) + shape)
    a[0] = np.abs(a[0]) + 0.02
    return a


@pytest.mark.parametrize("precision", ["float32", "float64"])
@pytest.mark.parametrize("n,shape,bc,curvature,fast", [
    (1, (2, 3, 5), (P, P, P), 1.0, True), (2, (1, 15, 31), (P, P, P), 0.5, False), (3, (3, 16, 32), (N, P, P), 1.0, True),
    (3, (5, 17, 33), (D, N, P), 0.4, False), (4, (40, 33, 34), (N, N, N), 1.0, False),
    (5, (7, 31, 65), (P, D, N), 0.0, True), (6, (300, 5, 6), (P, P, P), 1.0, True), (7, (6, 18, 30), (N, P, D), 0.5, True),
    (8, (9, 20, 40), (P, P, P), 0.5, False)])
def test_rhs_matches_oracle(n, shape, bc, curvature, fast, precision):
    p, og = build(shape, precision, bc, curvature=curvature, fast=fast)
    arr = phases(shape, n, n)
    u = torch.tensor(arr, dtype=p.vg.precision, device="cuda")
    assert p.fused_for(u)
    got = p.rhs(0.0, u).cpu().numpy()
    want = O.multiphase_ac_rhs(og.field(arr)[0], og, bc, eps=2.5, gab=1.2, M=0.8, curvature=curvature,
                               fast=fast).numpy()
    if n == 1:  # a single phase projects to 1 and does not move
        assert np.abs(got).max() <= 1e-6 * (1 if precision == "float32" else 1e-9)
        return
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err < TOL[precision], err


@pytest.mark.parametrize("precision", ["float32", "float64"])
@pytest.mark.parametrize("kind", ["dirichlet", "neumann"])
def test_staggered_rules(kind, precision):
    nodes = (9, 18, 35)
    bc = (D if kind == "dirichlet" else N, P, P)
    p, og = build(nodes, precision, bc, "staggered_x")
    arr = phases((nodes[0] - 2,) + nodes[1:], 3, 11)
    u = torch.tensor(arr, dtype=p.vg.precision, device="cuda")
    got = p.rhs(0.0, u)
    proj = p.project_to_simplex(u)
    lap = p.vg.laplace(p.pad_bc(proj))
    df = -lap + p.calc_potential_derivatives(proj)
    want = -p.M * p.gab * (df - df.mean(0, keepdim=True))
    err = float((got - want).norm() / want.norm())
    assert err < TOL[precision], err


@pytest.mark.parametrize("precision", ["float32", "float64"])
@pytest.mark.parametrize("stepper", [ForwardEuler, RungeKutta4])
def test_epilogues_equal_the_composition(stepper, precision):
    p, _ = build((11, 18, 35), precision, (N, P, P), curvature=0.5)
    u = torch.tensor(phases((11, 18, 35), 3, 3), dtype=p.vg.precision, device="cuda")
    dt = 0.05
    got = stepper(p, dt).step(0.0, u)
    if stepper is ForwardEuler:
        want = u + dt * p.rhs(0.0, u)
    else:
        k1 = p.rhs(0.0, u)
        k2 = p.rhs(0.0, u + 0.5 * dt * k1)
        k3 = p.rhs(0.0, u + 0.5 * dt * k2)
        k4 = p.rhs(0.0, u + dt * k3)
        want = u + (dt / 6) * (k1 + 2 * k2 + 2 * k3 + k4)
    assert torch.equal(got, want)


def test_replaced_rhs_is_not_bypassed():
    p, _ = build((5, 6, 7), "float64", (P, P, P))
    u = torch.rand((3, 5, 6, 7), dtype=torch.float64, device="cuda")
    p.rhs = lambda t, v: torch.ones_like(v)
    assert not p.fused_for(u)
    assert torch.equal(ForwardEuler(p, 0.5).step(0.0, u), u + 0.5)
