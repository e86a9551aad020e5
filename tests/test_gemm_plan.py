"""The default plan of the prefill GEMM (host side, CPU): which tile a shape runs
on. Kinds: 0 bf16, 1 SwiGLU, 2 int32, 3 dequant, 4 dequant SwiGLU, 5 bias, 6
bias + GELU; tiles 0-10 the ring kernel's, from 11 on the K-splitting one's."""

from __future__ import annotations

import pytest

import pytest

from ppu_amd import _lib


def test_refused_sizes():
    plan = _lib.load().q35_gemm_plan
    assert plan(0, 8, 64, 0) == plan(8, 0, 64, 0) == plan(8, 8, 0, 0) == -1
    assert plan(8, 8, 96, 0) == plan(8, 8, 64, 2) == plan(8, 8, 64, 7) == plan(8, 8, 64, -1) == -1
    assert plan(8, 8, 64, 0) >= 0 and plan(8, 8, 128, 2) >= 0


@pytest.mark.parametrize("kind,m,n", [(0, 441, 9456), (2, 441, 9456), (1, 4780, 4888), (4, 1299, 7664), (0, 8838, 5128)])
def test_widest_tile_from_16_stages(kind, m, n):
    """256x256 needs 16 stages of 128 bytes to pay for its prologue and epilogue."""
    plan = _lib.load().q35_gemm_plan
    stage = 128 if kind in (2, 3, 4) else 64
    assert all(plan(m, n, stage * nk, kind) not in (9, 10) for nk in range(1, 16))


def test_widest_tile_for_whole_rounds():
    plan = _lib.load().q35_gemm_plan
    assert plan(8192, 2048, 6144, 0) == 10 and plan(4000, 4090, 1024, 0) == 10
    assert plan(4000, 4090, 2048, 1) == 9 and plan(8192, 2048, 6144, 3) == 9


@pytest.mark.parametrize("m", [200, 256])
def test_int32_of_wide_outputs_leaves_the_ksplit_kernel(m):
    """Outputs wider than 4096 take the K-splitting kernel up to 128 operand rows
    only (64 x 96 tiles were slower than one round of the ring's)."""
    plan = _lib.load().q35_gemm_plan
    assert plan(m, 5120, 2048, 2) < 11 and plan(160, 5120, 2048, 2) >= 11
    assert plan(m, 2048, 2048, 2) >= 11 and plan(m, 5120, 2048, 0) >= 11
