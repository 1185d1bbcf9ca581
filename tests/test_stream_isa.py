"""ISA guard for what comes by LDS-DMA beside counted waits: hipcc waits for all that is in flight ahead of a load's first use, so
no load to registers may follow the first piece but those of a rare end."""
import re
import shutil

import pytest

from test_ppp_isa import KERNELS_LIB, OBJDUMP, subprocess


@pytest.mark.skipif(not OBJDUMP.exists() or not KERNELS_LIB.exists(), reason="llvm-objdump or the built library missing")
def test_index_rows_norms_and_masks_come_by_the_stream(tmp_path):
    lib = tmp_path / KERNELS_LIB.name
    shutil.copy(KERNELS_LIB, lib)
    subprocess.run([str(OBJDUMP), "--offloading", str(lib)], capture_output=True, check=True, cwd=tmp_path)
    found = {"knn_stream_kernel": 0, "knn_stream_floats_kernel": 0}
    for obj in sorted(tmp_path.glob(lib.name + ".*gfx950")):
        dis = subprocess.run([str(OBJDUMP), "-d", str(obj)], capture_output=True, text=True, check=True).stdout
        parts = re.split(r"\n[0-9a-f]+ <([^>]+)>:\n", dis)
        for name, body in zip(parts[1::2], parts[2::2]):
            for kernel in found:
                if kernel in name:
                    found[kernel] += 1
                    at = body.index("global_load_lds_dword")
                    assert not re.search(r"\sglobal_load_(?!lds)", body[at:]), name
                    assert not re.search(r"\sscratch_(load|store)", body), name
            assert "knn_stream" not in name or any(kernel in name for kernel in found), name
    assert found == {"knn_stream_kernel": 20, "knn_stream_floats_kernel": 10}
