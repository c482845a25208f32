"""Wavefronts per SIMD of the kernels that large systems are bound by, as the compiler reports them: the
FP32-multigrid PCG's product runs unfolded above 2,048 blocks and carries none of the fold's registers
there (45.8 us at 1,310,720 complex rows with them, 39.2 without)."""
import os
import re
import shutil
import subprocess

import pytest

from metriko_amd import build as B


@pytest.mark.slow
def test_unfolded_product_keeps_its_wavefronts(tmp_path):
    hipcc = shutil.which(B.HIPCC)
    if not hipcc:
        pytest.skip("no hipcc")
    flags = [f for f in B.FLAGS if f not in ("-Wall", "-fPIC")]
    r = subprocess.run([hipcc, *flags, "--offload-device-only", "-c", os.path.join(B.CSRC, "kernels.hip"), "-o",
                        str(tmp_path / "k.o"), "-Rpass-analysis=kernel-resource-usage"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    waves, name = {}, None
    for line in r.stderr.splitlines():
        if m := re.search(r"Function Name: (\S+)", line):
            name = m.group(1)
        elif m := re.search(r"Occupancy \[waves/SIMD\]: (\d+)", line):
            waves[name] = int(m.group(1))
    get = lambda cplx: [w for k, w in waves.items() if k.startswith(f"_ZN2mk8cgm_spmvILb{cplx}ELb0E")]  # noqa: E731
    assert len(get(1)) == 1 and get(1)[0] >= 6 and len(get(0)) == 1 and get(0)[0] >= 7
