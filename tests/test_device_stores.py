"""CPU check of the gfx950 assembly of every source with device code, compiled
as the Makefile does: whatever writes memory is a vector or an LDS instruction.
The check is by an allow-list over all instructions that store, exchange or
write back."""
import glob
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "mp-citdse_amd")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
WRITERS = re.compile(r"store|atomic|write|cmpst|swap|cache|_wb|_inc_|_dec_|"
                     r"_add_u|_sub_u|_min_|_max_|_or_b|_and_b|_xor_b")
MEMORY = re.compile(r"^(global|buffer|flat|scratch|ds|s)_")
ALLOWED = re.compile(r"^(global|buffer|flat|scratch)_(store|atomic)_|^ds_|"
                     r"^buffer_(wbl2|inv)$")
# scalar-unit instructions on registers whose names match WRITERS
SCALAR_ALU = re.compile(r"^s_(add|sub|min|max|or|and|xor)_[a-z]*[0-9]+$|"
                        r"^s_(and|or|xor)_saveexec_b64$|^s_swappc_b64$")


def sources():
    return sorted(os.path.basename(f)
                  for f in glob.glob(os.path.join(PKG, "csrc", "*.hip")))


def test_all_sources_are_looked_at():
    assert sources() == ["ci.hip", "engine.hip", "kernels.hip",
                         "persistent.hip"]


@pytest.mark.parametrize("src", sources())
def test_memory_is_written_by_vector_instructions(tmp_path, src):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    out = str(tmp_path / (src + ".s"))
    extra = ["-mllvm", "-disable-machine-licm"] if src == "persistent.hip" else []
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17",
                    "--cuda-device-only", "-S", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", *extra,
                    os.path.join(PKG, "csrc", src), "-o", out],
                   check=True, capture_output=True, timeout=300)
    with open(out) as f:
        ops = set(re.findall(r"^\s+([a-z][a-z0-9_]+)(?:\s|$)", f.read(),
                             flags=re.M))
    writers = {o for o in ops if MEMORY.match(o) and WRITERS.search(o)}
    assert not {o for o in writers
                if not ALLOWED.match(o) and not SCALAR_ALU.match(o)}
    if src in ("kernels.hip", "persistent.hip"):
        assert any(o.startswith("global_store") for o in writers)
