"""What the compiled kernels must not hold, read from the disassembly of the built library's gfx950 code objects."""
import os
import re
import shutil
import subprocess

import pytest

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.fixture(scope="module")
def disassembly(tmp_path_factory):
    from memarch_amd import _lib
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    d = tmp_path_factory.mktemp("isa")
    shutil.copy(_lib.LIB_PATH, d / "libmce.so")
    subprocess.run([OBJDUMP, "--offloading", "libmce.so"], cwd=d, check=True, capture_output=True)
    objs = sorted(f for f in os.listdir(d) if f.endswith("gfx950"))
    assert len(objs) == 3, objs   # mce, induct, swiglu
    return "".join(subprocess.run([OBJDUMP, "-d", f], cwd=d, check=True, capture_output=True, text=True).stdout
                   for f in objs)


def test_no_kernel_writes_back_the_l2(disassembly):
    """A device-scope release (buffer_wbl2) writes back the whole XCD's L2 from every wave that runs it. Kernels hand
    values on within a workgroup (barriers) or from launch to launch, so none needs one."""
    held, kernel = set(), None
    for line in disassembly.splitlines():
        m = re.match(r"[0-9a-f]+ <(.*)>:", line)
        if m:
            kernel = m.group(1)
        elif "buffer_wbl2" in line:
            held.add(kernel)
    assert kernel is not None and "v_mfma_f32_32x32x16_bf16" in disassembly
    assert not held, held
