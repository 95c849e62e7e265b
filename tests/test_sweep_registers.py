"""The register use of the ILU(0) sweeps, from the compiler's own report: a
wavefront that spills reads scratch memory between two barriers of every
level, which doubled the FP64 apply of rows with five to eight blocks."""
import os
import re
import subprocess

import pytest

from rhodst_amd import build


def test_sweeps_do_not_spill(tmp_path):
    try:
        hipcc = build._hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    r = subprocess.run([hipcc, *build.CFLAGS, "-x", "hip", "--cuda-device-only", "-Rpass-analysis=kernel-resource-usage",
                        "-c", os.path.join(build.CSRC, "solve.hip"), "-o", str(tmp_path / "solve.o")],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr
    use, name = {}, None
    for line in r.stderr.splitlines():
        if m := re.search(r"Function Name: (\S+)", line):
            name = m.group(1)
        elif m := re.search(r"ScratchSize \[bytes/lane\]: (\d+)", line):
            use[name] = int(m.group(1))
    sweeps = {k: v for k, v in use.items() if "k_stream_apply" in k or "k_tile_sweep" in k}
    assert len(sweeps) >= 12
    # 32 bytes: a handful of values outside the level loop
    assert all(v <= 32 for v in sweeps.values()), sweeps
