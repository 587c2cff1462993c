"""CPU emulation of the index arithmetic of the semi-implicit step's kernels and
of its adjoint's (tests/emulation/sweep_bounds.hip): the periodic Cahn-Hilliard
tile with its plane ring, the whole-plane sweeps, the line kernels at every
length they take, and the adjoint, through the geometry helpers that the
kernels and their launches use."""
import subprocess

import pytest

from tests.test_bounds_emulation import ROOT, hipcc


@pytest.mark.skipif(hipcc() is None, reason="hipcc is needed to build the host emulation")
def test_sweep_index_math_stays_in_bounds(tmp_path):
    exe = tmp_path / "sweep_bounds"
    cmd = [hipcc(), "-O2", "-std=c++17", "--offload-arch=gfx950", "-I", str(ROOT / "include"),
           "-I", str(ROOT / "evoxels_amd" / "csrc"), str(ROOT / "tests" / "emulation" / "sweep_bounds.hip"),
           "-o", str(exe)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    print(run.stdout)
    assert run.returncode == 0, run.stdout + run.stderr
    lines = run.stdout.strip().splitlines()
    assert len(lines) == 31 and all(line.startswith("OK ") for line in lines)
