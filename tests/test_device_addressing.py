"""The x-pass waits for its prefetched rows by the number of vector memory
operations that may still be under way.  That number means something for
global accesses only, so no x-pass kernel of the built library may hold a FLAT
access (a pointer of unknown address space, as one read from a table in memory
is to the compiler)."""
import os
import re
import shutil
import subprocess

import pytest

from helpers import PKG_DIR

LIB = os.path.join(PKG_DIR, "libchanflow.so")
OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")


@pytest.mark.skipif(not os.path.exists(OBJDUMP) or not os.path.exists(LIB), reason="no objdump or no built library")
def test_xpass_kernels_hold_no_flat_access(tmp_path):
    lib = shutil.copy(LIB, tmp_path)                  # the code objects are written beside it
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, stdout=subprocess.DEVNULL)
    seen = 0
    for name in sorted(os.listdir(tmp_path)):
        if not name.endswith("gfx950"):
            continue
        path = os.path.join(tmp_path, name)
        syms = subprocess.run([OBJDUMP, "-t", path], check=True, capture_output=True, text=True).stdout
        kernels = sorted(set(re.findall(r"\.text\s.*?(_Z\d+k_xpass_w\w*)$", syms, re.M)))
        if not kernels:
            continue
        asm = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--disassemble-symbols=" + ",".join(kernels), path],
                             check=True, capture_output=True, text=True).stdout
        flat = {}
        for head, body in re.findall(r"<(_Z\d+k_xpass_w\w*)>:\n(.*?)(?=\n\n|\Z)", asm, re.S):
            seen += 1
            assert "global_store" in body, head
            if n := len(re.findall(r"\bflat_(?:load|store|atomic)", body)):
                flat[head] = n
        assert not flat
    assert seen > 80                                  # batched and single, linearized and not, every length
