"""fp32 results of the persistent prompt GEMM (pgemm.hip, pgemm_ppp32_kernel)."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest
import torch

from copilot_for_consensus_amd._build import KERNELS_LIB
from copilot_for_consensus_amd.models.projection import Projection
from copilot_for_consensus_amd.ops import kernels as K

OBJDUMP = Path("/opt/rocm/lib/llvm/bin/llvm-objdump")


@pytest.mark.skipif(not OBJDUMP.exists() or not KERNELS_LIB.exists(), reason="llvm-objdump or the built library missing")
def test_store_count_matches_its_vmcnt_waits(tmp_path):
    """Its next tile's first waits keep 32 stores outstanding: exactly 32 in the interior (and 32 on the edge path), no scratch."""
    lib = tmp_path / KERNELS_LIB.name
    shutil.copy(KERNELS_LIB, lib)
    subprocess.run([str(OBJDUMP), "--offloading", str(lib)], capture_output=True, check=True, cwd=tmp_path)
    found = 0
    for obj in sorted(tmp_path.glob(lib.name + ".*gfx950")):
        dis = subprocess.run([str(OBJDUMP), "-d", str(obj)], capture_output=True, text=True, check=True).stdout
        parts = re.split(r"\n[0-9a-f]+ <([^>]+)>:\n", dis)
        for name, body in zip(parts[1::2], parts[2::2]):
            if "pgemm_ppp32_kernel" in name:
                found += 1
                assert len(re.findall(r"\sglobal_store_dwordx4\s", body)) == 64
                assert not re.search(r"\sglobal_store_(dword|dwordx2|dwordx3|short|byte)\s", body)
                assert not re.search(r"\s(scratch_(load|store)|buffer_store)", body)
    assert found == 1


@pytest.mark.gpu
@pytest.mark.parametrize("M, N, Kd", [(1, 64, 128), (255, 320, 192), (256, 256, 128), (700, 4096, 256), (4500, 4096, 192),
                                      (5130, 4160, 448)])
def test_equals_the_one_tile_kernel(M, N, Kd):
    """The same sums in the same order as the kernel of one tile per workgroup; edge tiles, odd and even K-tiles, one to
    three tiles per workgroup, rows of a wider result untouched."""
    g = torch.Generator("cuda").manual_seed(M)
    x = torch.randn(M, Kd, device="cuda", generator=g).bfloat16()
    w = Projection((torch.randn(N, Kd, device="cuda", generator=g) * 0.1).bfloat16()).packed
    want = K.pgemm(x, w, "f32", variant="pp")
    got = torch.full((M + 1, N), 7.0, device="cuda")
    K.pgemm(x, w, "f32", out=got[:M], variant="ppp")
    assert torch.equal(got[:M], want) and (got[M] == 7.0).all()
    exact = x.double() @ K._rowmajor(w).double().t()
    tol = Kd * 2.0 ** -24 * (x.double().abs() @ K._rowmajor(w).double().abs().t())
    assert ((want.double() - exact).abs() <= tol + 1e-30).all()
