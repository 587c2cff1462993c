"""CPU emulation of the explicit kernels' index arithmetic
(tests/emulation/explicit_bounds.hip) with the tile and chunk helpers that the
kernels use, in both types, at the edges of the tiles and of the chunks."""
import subprocess

import pytest

from tests.test_bounds_emulation import ROOT, hipcc


@pytest.mark.skipif(hipcc() is None, reason="hipcc is needed to build the host emulation")
def test_explicit_index_math_stays_in_bounds(tmp_path):
    exe = tmp_path / "explicit_bounds"
    cmd = [hipcc(), "-O2", "-std=c++17", "--offload-arch=gfx950", "-I", str(ROOT / "include"),
           "-I", str(ROOT / "evoxels_amd" / "csrc"), str(ROOT / "tests" / "emulation" / "explicit_bounds.hip"),
           "-o", str(exe)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(run.stdout)
    assert run.returncode == 0, run.stdout + run.stderr
    lines = run.stdout.strip().splitlines()
    assert len(lines) == 45 and all(line.startswith("OK ") for line in lines)
