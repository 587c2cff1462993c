"""The periodic Cahn-Hilliard right-hand-side tile inside the semi-implicit
step, against the float64 oracle: grids smaller than the stencil, one point
around the tile edges in y and z, x lengths around the short chunk and its
warm-up, several channels with their own parameters, and a grid large enough
for the wide float32 tile."""
import numpy as np
import pytest
import torch

import evoxels_amd as evx
from evoxels_amd.inversion import CHImexEngine
from evoxels_amd.voxelgrid import VoxelGridHip
from oracle import evoxels_oracle as O

pytestmark = pytest.mark.gpu

P3 = (("periodic", None),) * 3
SHAPES = [(1, 1, 1), (1, 2, 3), (2, 3, 5), (3, 15, 31), (4, 16, 32), (5, 17, 33), (6, 33, 63), (7, 18, 64), (9, 34, 65),
          (64, 5, 100), (300, 16, 34), (16, 1024, 1024)]


@pytest.mark.parametrize("precision", ["float32", "float64"])
@pytest.mark.parametrize("shape", SHAPES)
def test_step_matches_oracle(shape, precision):
    big = np.prod(shape) > 1e6
    if big and precision == "float64":
        pytest.skip("the wide tile is float32's")
    c = 1 if big else 3
    vf = evx.VoxelFields(shape, tuple(s * n for s, n in zip((1.0, 1.2, 0.9), shape)))
    vf.precision = precision
    vg = VoxelGridHip(vf.grid_info(), precision=precision, device="cuda")
    rng = np.random.default_rng(sum(shape))
    arr = 0.5 + 0.3 * rng.standard_normal((c,) + shape)  # values outside [0, 1]: the clip is active
    par = np.stack([np.linspace(2.0, 3.0, c), np.linspace(0.8, 1.3, c)], 1)
    eng = CHImexEngine(vg, c, 0.01)
    u = torch.tensor(arr, dtype=vg.precision, device="cuda")
    got = eng.step(u, eng.params(par)).cpu().double().numpy()
    og = O.OracleGrid(shape, vf.spacing, "float64")
    k2 = O.rfft_k_squared(shape, vf.spacing)
    for i in range(c):
        eps, D = par[i]
        u0 = u[i:i + 1].cpu().double()
        ref = O.imex_step(u0, lambda t, v: O.ch_rhs(v, og, P3, eps, D), O.imex_prefac(0.01, O.ch_symbol(k2, eps, D)))
        up = (ref - u0).numpy()[0]
        # the update: its right-hand side and transforms round at the size of the largest mu and flux
        tol = 5e-6 if precision == "float32" else 1e-13
        err = np.linalg.norm(got[i] - ref.numpy()[0]) / (np.linalg.norm(up) + 0.05 * np.linalg.norm(ref.numpy()))
        assert err < tol, (shape, i, err)
