"""Registers and scratch of the prefill attention's kernels, from the metadata of
the built gfx950 code object (LLVM tools on this build's own output): none keeps
anything in scratch, and those of 8 and 16 waves leave room for 4 waves per
SIMD (at most 128 registers of 512), which their tile sizes count on.  CPU only."""
import os
import re
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HSACO = os.path.join(ROOT, "rust-fp4-blackwell_amd", "build", "kernels.hsaco")
LLVM = "/opt/rocm/llvm/bin"


def test_prefill_attention_registers():
    if not os.path.exists(HSACO) or not os.path.exists(LLVM):
        pytest.skip("code object not built")
    with tempfile.TemporaryDirectory() as d:
        elf = os.path.join(d, "k.elf")
        subprocess.run([f"{LLVM}/clang-offload-bundler", "--unbundle", "--type=o",
                        "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--input={HSACO}", f"--output={elf}"], check=True)
        notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", elf], check=True, capture_output=True, text=True).stdout
    seen = 0
    for block in re.split(r"\n\s+- (?=\.agpr_count)", notes)[1:]:
        f = dict(re.findall(r"\.(name|vgpr_count|private_segment_fixed_size|max_flat_workgroup_size):\s+(\S+)", block))
        if not f["name"].startswith("rfp4_attn_prefill_"):
            continue
        seen += 1
        assert f["private_segment_fixed_size"] == "0", f
        if int(f["max_flat_workgroup_size"]) > 256:
            assert int(f["vgpr_count"]) <= 128, f
    assert seen == 44
