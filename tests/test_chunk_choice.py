"""The chunk length of the streaming kernels, computed on the host by every
launch (tests/emulation/chunk_choice.hip): the same as by looking at every
chunk count, in a small part of a launch's time also on grids of one tile and
a million planes."""
import subprocess

import pytest

from tests.test_bounds_emulation import ROOT, hipcc


@pytest.mark.skipif(hipcc() is None, reason="hipcc is needed to build the host program")
def test_chunk_choice(tmp_path):
    exe = tmp_path / "chunk_choice"
    cmd = [hipcc(), "-O2", "-std=c++17", "--offload-arch=gfx950", "-I", str(ROOT / "include"),
           "-I", str(ROOT / "evoxels_amd" / "csrc"), str(ROOT / "tests" / "emulation" / "chunk_choice.hip"),
           "-o", str(exe)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(run.stdout)
    assert run.returncode == 0, run.stdout + run.stderr
    lines = run.stdout.strip().splitlines()
    assert len(lines) == 4 and all(line.startswith("OK ") for line in lines)
