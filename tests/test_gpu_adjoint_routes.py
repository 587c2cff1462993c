"""The Cahn-Hilliard adjoint on thin grids, against autograd through the
float64 oracle: x axes cut into more than 64 chunks, and the separate kernels
that grids of few planes or rows take."""
import ctypes as C

import numpy as np
import pytest
import torch

from evoxels_amd import _lib
from evoxels_amd.inversion import CHImexEngine
from tests.test_gpu_adjoint import grid_for, oracle_step_autograd, rel

from tests.test_gpu_adjoint_stream import test_tile_edges as against_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["float64", "float32"])
@pytest.mark.parametrize("shape,c,based", [((300, 2, 3), 1, True), ((2001, 9, 5), 2, False), ((4000, 1, 70), 1, True)])
def test_more_than_64_chunks(shape, c, based, precision):
    against_oracle(shape, c, based, precision)


THIN = [((1, 600, 601), 4, True), ((2, 512, 512), 3, False), ((600, 1, 65), 16, True), ((1000, 3, 130), 7, False)]


def is_separate(shape, c, precision):
    g = _lib.make_grid((c,) + shape, (1.0,) * 3, (1.0,) * 3)
    n = C.c_size_t()
    code, size = (_lib.EVX_F32, 4) if precision == "float32" else (_lib.EVX_F64, 8)
    _lib.check(_lib.load().evx_ch_rhs_vjp_workspace_bytes(code, C.byref(g), C.byref(n)))
    return n.value >= 3 * size * c * int(np.prod(shape))


@pytest.mark.parametrize("precision", ["float64", "float32"])
@pytest.mark.parametrize("shape,c,based", THIN)
def test_separate_kernels(shape, c, based, precision):
    assert is_separate(shape, c, precision)
    against_oracle(shape, c, based, precision)


def test_separate_kernels_in_the_step():
    """The reverse step (prefactor term, in place on its cotangent) on a grid of
    one plane."""
    shape, c, dt = (1, 400, 400), 5, 0.1
    assert is_separate(shape, c, "float64")
    vf, vg = grid_for(shape, "float64", (1.0, 0.9, 1.1))
    rng = np.random.default_rng(3)
    arr = 0.5 + 0.3 * rng.standard_normal((c,) + shape)
    lam = rng.standard_normal(arr.shape)
    prm = np.stack([rng.uniform(2, 4, c), rng.uniform(0.5, 1.5, c)], 1)
    eng = CHImexEngine(vg, c, dt)
    par = eng.params(prm)
    u0 = torch.tensor(arr, device="cuda")
    u1 = eng.step(u0, par)
    lt = torch.tensor(lam, device="cuda")
    grads = []
    for inplace in (False, True):
        dp = torch.zeros((c, 2), dtype=torch.float64, device="cuda")
        lam0 = eng.step_vjp(u0, u1, lt.clone(), par, dp, None if inplace else torch.empty_like(lt))
        grads.append((lam0, dp))
    assert torch.equal(grads[0][0], grads[1][0]) and torch.equal(grads[0][1], grads[1][1])
    for k in range(c):
        u = torch.tensor(arr[k:k + 1], requires_grad=True)
        e, d = (torch.tensor(prm[k, i], dtype=torch.float64, requires_grad=True) for i in (0, 1))
        out = oracle_step_autograd(u, shape, vf.spacing, dt, e, d)
        want = torch.autograd.grad((out * torch.tensor(lam[k:k + 1])).sum(), (u, e, d))
        assert rel(grads[0][0][k:k + 1].cpu(), want[0]) < 1e-11
        # autograd differentiates the float32 prefactor in float32 arithmetic
        for i in range(2):
            size = float(torch.tensor(lam[k]).norm() * (out.detach() - u.detach()).norm()) / prm[k, i]
            assert abs(float(grads[0][1][k, i]) - float(want[1 + i])) < 2e-5 * size
