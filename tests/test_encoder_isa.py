"""The encoder's kernels ask for all they read at once: what they hold stays in registers, also where no norm takes it up."""
import re
import shutil

import pytest

from test_ppp_isa import KERNELS_LIB, OBJDUMP, subprocess

KERNELS = {"enc_tile_kernel": 6, "enc_ksplit_kernel": 4, "enc_norm_kernel": 1, "enc_gemm_kernel": 11}


@pytest.mark.skipif(not OBJDUMP.exists() or not KERNELS_LIB.exists(), reason="llvm-objdump or the built library missing")
def test_no_scratch(tmp_path):
    lib = tmp_path / KERNELS_LIB.name
    shutil.copy(KERNELS_LIB, lib)
    subprocess.run([str(OBJDUMP), "--offloading", str(lib)], capture_output=True, check=True, cwd=tmp_path)
    found = dict.fromkeys(KERNELS, 0)
    for obj in sorted(tmp_path.glob(lib.name + ".*gfx950")):
        dis = subprocess.run([str(OBJDUMP), "-d", str(obj)], capture_output=True, text=True, check=True).stdout
        parts = re.split(r"\n[0-9a-f]+ <([^>]+)>:\n", dis)
        for name, body in zip(parts[1::2], parts[2::2]):
            for k in KERNELS:
                if k in name:
                    found[k] += 1
                    assert not re.search(r"\sscratch_(load|store)", body), name
    assert found == KERNELS
