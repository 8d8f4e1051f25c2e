"""The register-before-retired check of test_asm_waits.py over the GEMM tile kernels."""
import os

import pytest

from _asm_waits import device_asm, inflight_uses, kernels
from test_asm_waits import CSRC, HIPCC, INCLUDE


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_no_tile_kernel_uses_a_register_before_its_load_retired():
    ks = kernels(device_asm(os.path.join(CSRC, "tile_gemm.hip"), [CSRC, INCLUDE], HIPCC))
    problems = [f"{name[:60]}: {p}" for name, instrs in ks.items() for p in inflight_uses(instrs)[:3]]
    assert len(ks) >= 4, "expected the tile kernels in the assembly"
    assert not problems, "\n".join(problems)
