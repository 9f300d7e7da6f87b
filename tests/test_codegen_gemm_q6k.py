"""The Q6_K instances of the fused GEMM keep the register and wait contract of
the others: no scratch, and hand-counted waits that match the loads emitted."""
import os

import pytest

import test_codegen as cg

pytestmark = pytest.mark.skipif(not os.path.exists(cg.HIPCC), reason="hipcc not found")


def test_gemm_q6k_wait_counts_and_registers(tmp_path):
    lines = cg._asm("gemm_q6k.hip", str(tmp_path / "gemm_q6k.s"))
    kernels = list(cg._gemm_kernels(lines))
    assert len(kernels) == 2, [k for k, _ in kernels]  # full and half tile
    bad = [(name, p) for name, body in kernels for p in [cg._gemm_wait_problems(body)] if p]
    assert not bad, bad
    assert not [l for l in lines if l.startswith("; ScratchSize:") and int(l.split()[-1])]
