"""Scratch of the N = 7 to 9 stage instances, from the compiler's resource report
(nekcem_amd/build.py's flags, device code only; nothing is run).  They
sit at 128 VGPRs, and what spilled there cost more than the kernel
before had gained: per-node materials 44 us against 41 at 9.9e5 nodes, with a
PML 90 against 68 (N = 9); with a dispersive region 65 against 62 (N = 8), the stages kept for the adjoint
115 against 102 at 2e6 nodes (N = 7)."""
import os
import re
import subprocess

import pytest

from nekcem_amd import build as B


def _report(tmp_path, n1):
    try:
        cc = B.hipcc()
    except RuntimeError:
        pytest.skip("needs hipcc")
    r = subprocess.run([cc] + B.HIPCC_FLAGS + ["-I", os.path.join(B.ROOT, "include"), "--cuda-device-only",
                                               "-Rpass-analysis=kernel-resource-usage", "-c", "-o",
                                               str(tmp_path / "o"), os.path.join(B.CSRC, f"order_n{n1}.hip")],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    out, key = {}, None
    for line in r.stderr.splitlines():
        m = re.search(rf"Function Name: _ZN3nkc10box_kernelILi{n1}ELi(\d)ELi(\d)ELi(\d)ELb(\d)ELi4ELi(\d)E", line)
        if "Function Name:" in line:
            key = tuple(map(int, m.groups())) if m else None
        m = re.search(r"ScratchSize \[bytes/lane\]: (\d+)", line)
        if m and key:
            out[key] = int(m.group(1))
    return out


def test_scratch_at_n9(tmp_path):
    scratch = _report(tmp_path, 10)    # (materials, mode, features, non-temporal, slabs) -> bytes a lane
    assert len(scratch) >= 20
    for nt in (0, 1):
        assert scratch[1, 0, 0, nt, 1] == 0          # per-node materials
        assert scratch[1, 0, 1, nt, 1] == 0          # with a source or a dispersive region
        for mat in (0, 1):
            assert scratch[mat, 0, 2, nt, 1] <= 32   # with a PML or an incident wave
            assert scratch[mat, 0, 3, nt, 1] <= 32   # with a sheet
            assert scratch[mat, 2, 0, nt, 1] == 0    # kept for the adjoint
            assert scratch[mat, 2, 1, nt, 1] <= 8


def test_scratch_at_n8(tmp_path):
    scratch = _report(tmp_path, 9)
    assert len(scratch) >= 16
    for mat in (0, 1):
        for nt in (0, 1):
            for feat in (0, 1, 2):
                assert scratch[mat, 0, feat, nt, 1] == 0


def test_scratch_of_kept_stages_at_n7(tmp_path):
    scratch = _report(tmp_path, 8)
    for mat in (0, 1):
        for nt in (0, 1):
            for feat in (0, 1):
                assert scratch[mat, 2, feat, nt, 1] == 0
