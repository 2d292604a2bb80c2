"""The generated code of xent_grad.hip, as test_kernel_invariants.py checks the other kernels whose
direct-to-LDS loads are issued from inline assembly: no spills, and no load whose scalar base a vector
instruction has written within the five wait states it needs."""
import os
import re
import subprocess

import pytest

from tests.test_kernel_invariants import HIPCC, ROOT


@pytest.fixture(scope="module")
def asm(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    out = tmp_path_factory.mktemp("asm") / "xent_grad.s"
    subprocess.run([HIPCC, "-x", "hip", "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-I", os.path.join(ROOT, "include"), "--cuda-device-only", "-S",
                    os.path.join(ROOT, "tritonops_amd", "csrc", "xent_grad.hip"), "-o", str(out)],
                   check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    return out.read_text()


def test_registers(asm):
    seen = 0
    for block in asm.split("- .agpr_count:")[1:]:
        seen += 1
        assert re.search(r"\.vgpr_spill_count:\s+0\b", block) and re.search(r"\.sgpr_spill_count:\s+0\b", block)
    assert seen == 4   # product and sum, bf16 and f16


def test_scalar_bases_are_not_fresh_vector_results(asm):
    lines = [l for l in asm.split("\n") if l.strip() and not l.strip().startswith((";", "."))]
    loads = 0
    for k, line in enumerate(lines):
        m = re.search(r"global_load_lds_dwordx4 v\d+, s\[(\d+):(\d+)\]", line)
        if not m:
            continue
        loads += 1
        base = set(range(int(m.group(1)), int(m.group(2)) + 1))
        for prev in reversed(lines[max(k - 6, 0):k]):
            if prev.strip().endswith(":"):
                break
            w = re.match(r"\s*v_\S+\s+s(?:\[(\d+):(\d+)\]|(\d+)\b)", prev)
            if w:
                lo = int(w.group(1) or w.group(3))
                assert not base & set(range(lo, int(w.group(2) or lo) + 1)), (prev.strip(), line.strip())
    assert loads >= 32
