"""What the grouped kernels are launched with, from the device code hipcc makes here: the experts' rows travel in the arguments of the kernels that
read them there, and of no others."""
import importlib.util
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "g-core-gh_amd", "csrc")


@pytest.mark.skipif(shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"), reason="needs hipcc")
def test_tables_travel_only_with_the_kernels_that_read_them(tmp_path):
    spec = importlib.util.spec_from_file_location("check_asm_operands", os.path.join(CSRC, "check_asm_operands.py"))
    C = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(C)
    out = tmp_path / "big.s"
    subprocess.run([C.HIPCC, *C.FLAGS, os.path.join(CSRC, "gemm_fp8_big.hip"), "-o", str(out)], check=True, capture_output=True)
    kernels = re.findall(r"\.amdhsa_kernel (\S*gemm_asm_grouped\S*)\n(?:(?!\.end_amdhsa_kernel).)*?\.amdhsa_kernarg_size (\d+)", out.read_text(), re.S)
    assert len(kernels) >= 14
    by_table = {"HostOffsets": [], "HostRows": [], "": []}
    for name, size in kernels:
        by_table[next((t for t in ("HostOffsets", "HostRows") if t in name), "")].append(int(size))
    assert len(by_table["HostOffsets"]) == 2 and len(by_table["HostRows"]) == 2
    assert all(2064 <= s <= 4096 for t in ("HostOffsets", "HostRows") for s in by_table[t])
    assert len(by_table[""]) >= 10 and max(by_table[""]) <= 512              # 256 of them the runtime's own
