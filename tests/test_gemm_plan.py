"""The default plan of the prefill GEMM (host side, CPU): which tile a shape runs
on. Kinds: 0 bf16, 1 SwiGLU, 2 int32, 3 dequant, 4 dequant SwiGLU, 5 bias, 6
bias + GELU; tiles 0-10 the ring kernel's, from 11 on the K-splitting one's."""

from __future__ import annotations

import pytest

from ppu_amd import _lib


def test_refused_sizes():
    plan = _lib.load().q35_gemm_plan
    assert plan(0, 8, 64, 0) == plan(8, 0, 64, 0) == plan(8, 8, 0, 0) == -1
    assert plan(8, 8, 96, 0) == plan(8, 8, 64, 2) == plan(8, 8, 64, 7) == plan(8, 8, 64, -1) == -1
    assert plan(8, 8, 64, 0) >= 0 and plan(8, 8, 128, 2) >= 0
