"""The decode attention kernels are to fit eight waves on a SIMD, with the new token's rotary embedding inside as well: launches that just
fit one round of eight workgroups per compute unit go into a second one otherwise.  Read off the compiler's report (no GPU)."""
import re
import shutil
import subprocess

import pytest


@pytest.mark.skipif(not (shutil.which("hipcc") or shutil.which("/opt/rocm/bin/hipcc")), reason="no hipcc")
def test_eight_waves(tmp_path):
    from flh_amd.csrc import build
    flags = [f for f in build.FLAGS if f not in ("-shared", "-fPIC")]
    r = subprocess.run([shutil.which("hipcc") or "/opt/rocm/bin/hipcc", *flags, *build.VGPR_FORM, "--cuda-device-only",
                        "-Rpass-analysis=kernel-resource-usage", "-c", str(build.HERE / "decode_attention.hip"),
                        "-o", str(tmp_path / "x.o")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    kernels = re.findall(r"Function Name: (\S+).*?Occupancy \[waves/SIMD\]: (\d+)", r.stderr, re.S)
    partial = {name: int(waves) for name, waves in kernels if "decode_attention_partial" in name}
    assert len(partial) == 16 and all(w == 8 for w in partial.values()), partial
