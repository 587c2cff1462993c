"""The whole-plane z/y sweeps (square y-z planes) in the semi-implicit and the
exponential steps: every plane length in both types, with an odd number of planes
and one to three channels, against the float64 oracle and against the
runtime-radix sweeps; the sums their inverse leaves; x slabs."""
import math

import numpy as np
import pytest
import torch

import evoxels_amd as evx
from evoxels_amd import _lib
from evoxels_amd.problem_definition import CahnHilliard, ReactionDiffusion
from evoxels_amd.timesteppers import ExponentialEuler, PseudoSpectralIMEX
from evoxels_amd.voxelgrid import VoxelGridHip
from oracle import evoxels_oracle as O

pytestmark = pytest.mark.gpu

P3 = (("periodic", None),) * 3


@pytest.mark.parametrize("precision", ["float32", "float64"])
@pytest.mark.parametrize("n,nx,c", [(n, nx, c) for n in (32, 48, 64, 96, 100, 128)
                                    for nx, c in ((1, 3), (5, 1), (9, 2))]
                         + [(128, 46, 1), (128, 48, 1), (128, 25, 2)])  # 128 in float64: from 48 planes on
def test_square_planes(n, nx, c, precision):
    shape = (nx, n, n)
    vf = evx.VoxelFields(shape, tuple(s * k for s, k in zip((0.9, 1.1, 1.3), shape)))
    vf.precision = precision
    vg = VoxelGridHip(vf.grid_info(), precision=precision, device="cuda")
    arr = 0.5 + 0.08 * np.random.default_rng(n + nx).standard_normal((c,) + shape)
    u = torch.tensor(arr, dtype=vg.precision, device="cuda")
    og = O.OracleGrid(shape, vf.spacing, "float64")
    k2 = O.rfft_k_squared(shape, vf.spacing)
    # one step's roundings of a field of order one; the exponential multiplier is
    # a float32 table (2 ulp apart between CPU and GPU) times a small update
    for prob, cls, sym, rhs, tol in (
            (CahnHilliard(vg, eps=2.0, D=1.5), PseudoSpectralIMEX, O.ch_symbol(k2, 2.0, 1.5),
             lambda t, v: O.ch_rhs(v, og, P3, 2.0, 1.5), 1e-12),
            (ReactionDiffusion(vg, D=0.8), ExponentialEuler, O.rd_symbol(k2, 0.8),
             lambda t, v: O.rd_rhs(v, og, P3, 0.8), 2e-8)):
        step = cls(prob, 0.05)
        fast = step.step(0.0, u)
        plan, _ = step.workspace(u)
        lib = _lib.load()
        if c == 1:
            flags = torch.zeros(2, dtype=torch.int32, device="cuda")
            rec = step.last_step_sums(fast, flags)
            if rec is not None:
                exact = math.fsum(fast.cpu().double().numpy().ravel())
                assert abs(float(rec[0]) - exact) <= 1e-14 * abs(exact) and flags.tolist() == [0, 0]
            bad = u.clone()
            bad[0, nx // 2, n // 2, 3] = float("nan")
            if rec is not None:
                step.last_step_sums(step.step(0.0, bad), flags)
                assert flags.tolist()[0] == 1
        into = u.clone()
        step.step_into(into, into)
        assert torch.equal(into, fast)  # in place
        for opt, value, default in ((_lib.OPT_SPECIALIZED, 0, 1), (_lib.OPT_SLABS, 2, 0)):
            _lib.check(lib.evx_fft_plan_set_option(plan.handle, opt, value), "option")
            other = step.step(0.0, u)
            _lib.check(lib.evx_fft_plan_set_option(plan.handle, opt, default), "option")
            if opt == _lib.OPT_SLABS:
                assert torch.equal(other, fast)
            else:
                assert float((other - fast).abs().max()) < (1e-13 if precision == "float64" else 1e-5)
        pre = O.imex_prefac(0.05, sym) if cls is PseudoSpectralIMEX else O.etd1_multiplier(0.05, sym)
        for k in range(c):
            ref = O.imex_step(og.field(arr[k]), rhs, pre)[0].numpy()
            err = np.linalg.norm(fast[k].cpu().numpy() - ref) / np.linalg.norm(ref)
            assert err < (2e-6 if precision == "float32" else tol), (cls.__name__, k, err)
