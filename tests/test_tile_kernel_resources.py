"""Register, LDS and scratch budgets of the list passes over LDS tiles (CPU only:
the kernels are compiled to gfx950 assembly here).

A workgroup has 8 waves, two per SIMD, and a CU 512 VGPRs a lane per SIMD and 160
KiB of LDS, so these counts set how many workgroups share a CU: four of lambda
and of the vorticity pass (64 VGPRs, 40 KiB), three of the build and of delta-p
(80 VGPRs), two of XSPH (60 KiB).  Delta-p spills up to 16 bytes a lane."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# kernel (mangled-name fragment) -> largest allowed VGPRs, LDS and scratch bytes
BUDGET = {
    "k_tile_buildE": (80, 163840 // 3, 0),
    "k_tile_lambdaE": (64, 163840 // 4, 0),
    "k_tile_deltapILb0ELi4E": (80, 163840 // 3, 16),
    "k_tile_deltapILb1ELi4E": (80, 163840 // 3, 16),
    "k_tile_deltapILb0ELin1E": (80, 163840 // 3, 16),
    "k_tile_deltapILb1ELin1E": (80, 163840 // 3, 16),
    "k_tile_xsphE": (128, 163840 // 2, 0),
    "k_tile_vortE": (64, 163840 // 4, 0),
}


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="no hipcc")
def test_tiled_kernels_keep_their_budgets(tmp_path):
    import sys
    sys.path.insert(0, ROOT)
    from fluid_amd import build as B

    flags = [f for f in B.HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    out = str(tmp_path / "k.s")
    cmd = [B.hipcc(), *flags, "--cuda-device-only", "-S", "-I", os.path.join(ROOT, "include"),
           "-o", out, os.path.join(ROOT, "fluid_amd", "csrc", "pbf_kernels.hip")]
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
                       timeout=600)
    assert r.returncode == 0, r.stdout[-3000:]
    asm = open(out).read()
    found = {}
    for m in re.finditer(r"\.amdhsa_kernel (\S+)\n(.*?)\.end_amdhsa_kernel", asm, re.S):
        for frag in BUDGET:
            if frag in m.group(1) and "GLOBAL__N_" in m.group(1):
                found[frag] = tuple(
                    int(re.search(rf"\.amdhsa_{k} (\d+)", m.group(2)).group(1))
                    for k in ("next_free_vgpr", "group_segment_fixed_size",
                              "private_segment_fixed_size"))
    assert set(found) == set(BUDGET), sorted(set(BUDGET) - set(found))
    over = {k: (v, BUDGET[k]) for k, v in found.items()
            if any(a > b for a, b in zip(v, BUDGET[k]))}
    assert not over, over
