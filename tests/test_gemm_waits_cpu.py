"""The matrix product that loads straight into LDS (gemm_tn8_kernel) waits for its
own LDS reads before every barrier that lets other waves overwrite what they read:
read from the assembly of a build made here."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_lds_reads_return_before_the_barrier(tmp_path):
    src, out = tmp_path / "gemm.hip", tmp_path / "gemm.s"
    src.write_text('#include "%s/gaga_amd/csrc/xcs_mfma.h"\n'
                   "template __global__ void xcs::gemm_tn8_kernel<xcs::FMT_BF16>(xcs::GemmArgs);\n"
                   "template __global__ void xcs::gemm_tn8_kernel<xcs::FMT_FP8>(xcs::GemmArgs);\n" % ROOT)
    subprocess.check_call([HIPCC, "-O3", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature",
                           "-Xclang", "-packed-fp32-ops", "--cuda-device-only", "-S", "-o", str(out), str(src)],
                          stderr=subprocess.DEVNULL)
    kernels = re.findall(r"^(_Z\S*gemm_tn8_kernel\S*):(.*?)s_endpgm", out.read_text(), re.S | re.M)
    assert len(kernels) == 2
    for name, body in kernels:
        ops = [l.split(";")[0].strip() for l in body.splitlines()]
        ops = [l for l in ops if l and not l.startswith((".", "#")) and not l.endswith(":")]
        at = [i for i, l in enumerate(ops) if l.startswith("s_barrier")]
        assert at, name
        for i in at:
            waited = False
            for l in reversed(ops[:i]):
                if l.startswith("s_waitcnt") and "lgkmcnt(0)" in l:
                    waited = True
                if waited or l.startswith(("ds_read", "v_mfma", "s_cbranch", "s_branch")):
                    break
            assert waited, (name, ops[max(0, i - 4):i + 1])
