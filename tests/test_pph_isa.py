"""ISA guard for the persistent prompt GEMM's tiles of 192 and 224 rows, as tests/test_ppp_isa.py has it for 256: the interior
epilogue's stores are those that the next tile's first waits count, and nothing spills."""
import re

import pytest

from test_ppp_isa import KERNELS_LIB, OBJDUMP, subprocess
import shutil

# EPI -> what stores the interior block (a number per 16 rows) and the edge path (4 per 16 rows)
STORES = {"0": (2, "dwordx2"), "3": (1, "dword"), "4": (4, "dwordx4"), "5": (1, "dword"), "6": (2, "dwordx2")}


@pytest.mark.skipif(not OBJDUMP.exists() or not KERNELS_LIB.exists(), reason="llvm-objdump or the built library missing")
def test_store_counts_match_the_waits(tmp_path):
    lib = tmp_path / KERNELS_LIB.name
    shutil.copy(KERNELS_LIB, lib)
    subprocess.run([str(OBJDUMP), "--offloading", str(lib)], capture_output=True, check=True, cwd=tmp_path)
    bodies = {}
    for obj in sorted(tmp_path.glob(lib.name + ".*gfx950")):
        dis = subprocess.run([str(OBJDUMP), "-d", str(obj)], capture_output=True, text=True, check=True).stdout
        parts = re.split(r"\n[0-9a-f]+ <([^>]+)>:\n", dis)
        for name, body in zip(parts[1::2], parts[2::2]):
            if m := re.search(r"pgemm_pph_kernelILi(\d)ELi(\d)E", name):
                bodies[m.groups()] = body
    assert set(bodies) == {(e, h) for e in STORES for h in "67"}, sorted(bodies)
    for (epi, mt), body in bodies.items():
        per, edge = STORES[epi]
        want = {"dwordx4": per * int(mt), "dwordx2": 0, "dword": 0}
        want[edge] += 4 * int(mt)
        got = {op: len(re.findall(r"\sglobal_store_" + op + r"\s", body)) for op in want}
        assert got == want, (epi, mt, got)
        assert not re.search(r"\sscratch_(load|store)|\sbuffer_store", body), (epi, mt)
