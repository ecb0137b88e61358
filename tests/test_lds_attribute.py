"""Kernels launched with dynamic LDS past the default limit need an attribute
call of their own: the library holds one flag for each of them, not one for each
signature (which both head sizes' attention, and the f16 GEMM's epilogues,
share)."""
import re
import shutil
import subprocess

import pytest

from nemo_amd import _lib


@pytest.mark.skipif(shutil.which("nm") is None, reason="needs binutils")
def test_every_dynamic_lds_kernel_has_its_own_flag():
    names = [line.split()[-1] for line in subprocess.check_output(["nm", _lib.LIB_PATH], text=True).splitlines()]
    # name and template arguments, as a flag's name holds them too
    kernel = re.compile(r"_ZN4nemo(\d+(?:gemm_big|gemm_wide|gemm_f16|attention)_kernelI\w+?E)EvP")
    kernels = {m.group(1) for m in map(kernel.match, names) if m}
    assert {"16attention_kernelILi64EE", "16attention_kernelILi128EE"} <= kernels
    flags = [n for n in names if "9allow_lds" in n and n.endswith("4done")]
    without = [n for n in kernels if not any(n in f for f in flags)]
    assert not without, f"{len(without)} of {len(kernels)} kernels have none, such as {without[0]}"
    assert len(flags) == len(kernels)
