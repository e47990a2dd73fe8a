"""What one lane leaves in LDS for another is read behind a barrier: looked for in the device code that the compiler makes of the source, because a
read that overtakes the write need not show in any one run."""
import importlib.util
import os
import re
import shutil
import subprocess

import pytest

from conftest import ROOT


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs the compiler")
@pytest.mark.parametrize("half", [False, True])
def test_list_of_tokens(half, tmp_path):
    """dK/dV: a barrier stands between the last 16-bit store (the list's entries are the only ones) and the first read that follows it."""
    spec = importlib.util.spec_from_file_location("build_script", os.path.join(ROOT, "infllmv2_cuda_impl_amd", "csrc", "build.py"))
    script = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(script)
    asm = tmp_path / "dkdv.s"
    subprocess.run(["hipcc", *script.HIPCC_FLAGS, *(["-DIV2_F16=1"] if half else []), "-I", script.include_dir(), "--cuda-device-only", "-S",
                    os.path.join(script.CSRC, "stage2_bwd_dkdv.hip"), "-o", str(asm)], check=True, stderr=subprocess.DEVNULL)
    kernels = re.findall(r"^(_Z\w*bwd_dkdv_wave_kernel\w*):(.*?)^\.Lfunc_end", asm.read_text(), re.M | re.S)
    assert kernels
    for name, body in kernels:
        ops = re.findall(r"^\s+(ds_write_b16|ds_read\w*|s_barrier)\b", body, re.M)
        behind = ops[len(ops) - ops[::-1].index("ds_write_b16"):]
        assert behind[0] == "s_barrier", name
