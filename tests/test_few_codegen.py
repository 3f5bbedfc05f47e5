"""The few-token GEMM's compiled form: no kernel of it spills, and none holds a packed FP32
instruction."""
import os
import re
import subprocess

from apeiron_amd import build


def test_few_token_kernels_do_not_spill(tmp_path):
    out = str(tmp_path / "few.s")
    flags = [f for f in build.FLAGS if f not in ("-shared",)]
    subprocess.run([build.HIPCC, *flags, "-x", "hip", "--cuda-device-only", "-S", os.path.join(build.CSRC, "ah_few.hip"), "-o", out],
                   check=True, capture_output=True)
    asm = open(out).read()
    kernels = re.findall(r"\.amdhsa_kernel (\S*gemm_few_kernel\S*)(.*?)\.end_amdhsa_kernel", asm, re.S)
    assert len(kernels) == 24  # six families x one / two token tiles x with / without the SwiGLU epilogue
    for name, body in kernels:
        assert re.search(r"private_segment_fixed_size 0\b", body), name
    assert not re.search(r"\bv_pk_(add|mul|fma)_f32\b", asm)


def test_few_token_kernels_read_codes_whole(tmp_path):
    """Code rows at any byte are staged by whole dwords: no kernel loads a byte at a time from memory."""
    out = str(tmp_path / "few.s")
    flags = [f for f in build.FLAGS if f not in ("-shared",)]
    subprocess.run([build.HIPCC, *flags, "-x", "hip", "--cuda-device-only", "-S", os.path.join(build.CSRC, "ah_few.hip"), "-o", out],
                   check=True, capture_output=True)
    assert not re.search(r"\b(global|flat|buffer)_load_[us]byte", open(out).read())
