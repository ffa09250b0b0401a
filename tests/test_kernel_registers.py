"""No kernel of the library spills vector registers to memory: the tuned kernels are shaped by how many wavefronts share a SIMD's
registers, and a form that does not fit runs, correctly, at half the speed.  Read from the notes of the code objects built here."""
import os
import re
import shutil
import subprocess

import pytest

import innova_amd as ia

BIN = "/opt/rocm/llvm/bin/"
# one register of the serial chain's wavefront, stored once before its loop
ALLOWED = {"engine_kernel": 1}


@pytest.mark.skipif(not os.path.exists(BIN + "llvm-readelf"), reason="no object reader")
def test_no_kernel_spills_vector_registers(tmp_path):
    lib = shutil.copy(ia._lib.LIB_PATH, tmp_path)
    subprocess.run([BIN + "llvm-objdump", "--offloading", lib], cwd=tmp_path, check=True, capture_output=True)
    spills = {}
    for name in sorted(os.listdir(tmp_path)):
        if "gfx950" in name:
            notes = subprocess.run([BIN + "llvm-readelf", "--notes", name], cwd=tmp_path, check=True, capture_output=True, text=True).stdout
            spills.update((k, int(n)) for k, n in re.findall(r"\.name:\s+(_Z\S+).*?\.vgpr_spill_count:\s+(\d+)", notes, re.S))
    assert len(spills) > 100
    bad = {k: n for k, n in spills.items() if n > max((v for a, v in ALLOWED.items() if a in k), default=0)}
    assert not bad, bad
