"""Registers of the built few-token kernels, from the metadata of their code
object."""
import re
import shutil
import subprocess

import pytest

from conftest import ROOT

OBJ = ROOT / "qwen-rust-inference_amd" / "build" / "gemm_kw.o"
LLVM = "/opt/rocm/llvm/bin/"


@pytest.mark.skipif(not OBJ.exists() or not shutil.which(LLVM + "clang-offload-bundler"), reason="no built object here")
def test_few_token_accumulators_stay_out_of_agprs(tmp_path):
    """Every kernel of gemm_kw.hip asks for two waves per SIMD: 256 registers,
    none of them accumulation registers, and nothing spilled."""
    fat, co = tmp_path / "fat", tmp_path / "co"
    subprocess.run([LLVM + "llvm-objcopy", f"--dump-section=.hip_fatbin={fat}", str(OBJ), str(tmp_path / "o")], check=True)
    subprocess.run([LLVM + "clang-offload-bundler", "--unbundle", "--type=o", f"--input={fat}", f"--output={co}",
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
    notes = subprocess.run([LLVM + "llvm-readelf", "--notes", str(co)], check=True, capture_output=True, text=True).stdout
    kernels = re.findall(r"\.agpr_count:\s+(\d+).*?\.name:\s+(\S+).*?\.vgpr_count:\s+(\d+)\s+\.vgpr_spill_count:\s+(\d+)",
                         notes, re.S)
    assert len(kernels) == 21, len(kernels)  # 7 tiles in 3 formats
    for agprs, name, vgprs, spills in kernels:
        assert (int(agprs), int(spills)) == (0, 0) and int(vgprs) <= 256, (name, agprs, vgprs, spills)
