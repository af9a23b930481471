"""Register use of the fused steps, from the compiler's resource remarks (no GPU needed)."""
import re
import subprocess
from pathlib import Path

import pytest

from miniappsforhpe_amd import build as B


@pytest.mark.parametrize("src", ["fused_kernels.hip", "batch.hip"])
def test_fused_steps_spill_nothing(src, tmp_path):
    """Every form of the fused steps (snapshot mode, sponge) fits the 128 VGPRs that 16 waves a CU leave it: a spilled
    word is stored and loaded again in every plane and cost the FP16 image with a sponge 15%."""
    if not Path(B.HIPCC).exists():
        pytest.skip("no hipcc")
    r = subprocess.run([B.HIPCC, *B.HIP_FLAGS, "-Rpass-analysis=kernel-resource-usage", "--offload-device-only", "-c",
                        str(B.CSRC / src), "-o", str(tmp_path / "k.o")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    use = {n: (int(v), int(s)) for n, v, s in re.findall(
        r"Function Name: (\S*k_fused_\S*).*?ScratchSize[^:]*: (\d+).*?VGPRs Spill: (\d+)", r.stderr, re.S)}
    assert len(use) >= 16
    assert {n: v for n, v in use.items() if v != (0, 0)} == {}
