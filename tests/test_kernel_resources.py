"""The fused Euler kernels as the compiler lays them out for gfx950 (its own resource remarks): no vector
registers spilled, no scratch memory, and the occupancy that the launcher asks for is there."""
import os
import re
import shutil
import subprocess

import pytest

from hyperboliconvergence_amd import build


@pytest.mark.parametrize("basis,flux", [(1, 4), (0, 5)], ids=["primitive-ausmpup", "conserved-roe"])
def test_fused_kernels_spill_nothing(tmp_path, basis, flux):
    if not shutil.which(build.HIPCC):
        pytest.skip("no hipcc")
    cmd = next(c for o, c in build._jobs() if os.path.basename(o) == f"stage_L1_B{basis}_F{flux}_P64.o")
    cmd = cmd[:-1] + [str(tmp_path / "k.o"), "--cuda-device-only", "-Rpass-analysis=kernel-resource-usage"]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    found = {}
    for block in r.stderr.split("Function Name: ")[1:]:
        name = block.split()[0]
        if "FusedTile" in name:
            found[name] = {k: int(re.search(rf"{k}[^:\n]*: (\d+)", block).group(1)) for k in ("ScratchSize", "VGPRs Spill")}
    assert len(found) == 13   # three shapes, uniform or not, folding or not, and the one with 64-bit offsets
    assert all(f == {"ScratchSize": 0, "VGPRs Spill": 0} for f in found.values()), found
    missed = [m for m in re.findall(r"failed to meet occupancy target[^\n]*", r.stderr) if "FusedTile" in m]
    assert not missed, missed
