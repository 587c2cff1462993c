"""The streaming Cahn-Hilliard adjoint at the edges of its tiles (64 voxels along
z, eight rows of them, x chunks) and on grids smaller than its halo of three,
against autograd through the float64 oracle."""
import numpy as np
import pytest
import torch

import evoxels_amd as evx
from evoxels_amd.inversion import ch_rhs_vjp
from evoxels_amd.voxelgrid import VoxelGridHip
from oracle import evoxels_oracle as O

pytestmark = pytest.mark.gpu

P3 = (("periodic", None),) * 3


@pytest.mark.parametrize("precision", ["float64", "float32"])
@pytest.mark.parametrize("shape,c,based", [((1, 1, 1), 1, True), ((2, 3, 1), 2, False), ((1, 2, 5), 1, True),
                                           ((4, 1, 200), 1, False), ((3, 8, 64), 2, True), ((5, 9, 65), 3, True),
                                           ((71, 7, 63), 1, True), ((9, 17, 130), 1, False), ((2, 300, 3), 1, True)])
def test_tile_edges(shape, c, based, precision):
    vf = evx.VoxelFields(shape, tuple(s * n for s, n in zip((0.9, 1.1, 1.3), shape)))
    vf.precision = precision
    vg = VoxelGridHip(vf.grid_info(), precision=precision, device="cuda")
    rng = np.random.default_rng(sum(shape))
    ut = torch.tensor(0.5 + 0.4 * rng.standard_normal((c,) + shape), dtype=vg.precision, device="cuda")
    ut.view(-1)[0] = 1.0  # a clip bound itself
    wt = torch.tensor(rng.standard_normal((c,) + shape), dtype=vg.precision, device="cuda")
    base = torch.tensor(rng.standard_normal((c,) + shape), dtype=vg.precision, device="cuda") if based else None
    eps, D = 2.5, 1.3
    grad, dp = ch_rhs_vjp(vg, ut, wt, eps, D, base=base)
    assert torch.equal(grad, ch_rhs_vjp(vg, ut, wt, eps, D, base=base)[0])
    og = O.OracleGrid(shape, vf.spacing, "float64")
    theta = (torch.tensor(eps, dtype=torch.float64), torch.tensor(D, dtype=torch.float64))
    # the parameter sums are held against the size of their terms
    tol_u, tol_p = (1e-12, 1e-11) if precision == "float64" else (2e-5, 2e-5)
    for k in range(c):
        u = ut[k:k + 1].cpu().double().requires_grad_(True)
        w = wt[k:k + 1].cpu().double()
        th = tuple(t.clone().requires_grad_(True) for t in theta)
        want = torch.autograd.grad((O.ch_rhs(u, og, P3, *th) * w).sum(), (u,) + th)
        gu = want[0] + (base[k:k + 1].cpu().double() if based else 0)
        err = float((grad[k:k + 1].cpu().double() - gu).norm())
        assert err <= tol_u * float(gu.norm()), err
        for j in range(2):
            v = tuple(torch.tensor(float(i == j), dtype=torch.float64) for i in range(2))
            dr = torch.autograd.functional.jvp(lambda e, d: O.ch_rhs(u.detach(), og, P3, e, d), theta, v)[1]
            assert abs(float(dp[k, j]) - float(want[1 + j])) <= tol_p * float(w.norm() * dr.norm())
