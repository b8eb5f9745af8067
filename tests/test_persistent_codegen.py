"""Code generation of the persistent kernels (CPU only), as compiled by the
Makefile: no out-of-line calls; the row kernels and the state save without a
private segment, the tile kernel with at most the few bytes its full register
file spills outside the sweep."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "mp-citdse_amd", "csrc", "persistent.hip")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def test_persistent_kernels(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    out = tmp_path / "persistent.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17",
                    "--cuda-device-only", "-S", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "-mllvm",
                    "-disable-machine-licm", SRC, "-o", str(out)],
                   check=True, capture_output=True, timeout=300)
    asm = out.read_text()
    assert "s_swappc_b64" not in asm and "s_setpc_b64" not in asm
    names = [n for n in re.findall(r"^\s+\.name:\s+(\S+)", asm, flags=re.M)
             if n.startswith("_Z")]
    priv = [int(p) for p in re.findall(
        r"^\s+\.private_segment_fixed_size:\s+(\d+)", asm, flags=re.M)]
    assert len(names) == len(priv) == 6
    for n, p in zip(names, priv):
        assert p <= (16 if "k_tiles_run" in n else 0), (n, p)
