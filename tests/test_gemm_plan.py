"""The default plan of the prefill GEMM (host side, CPU): which tile a shape runs
on. Kinds: 0 bf16, 1 SwiGLU, 2 int32, 3 dequant, 4 dequant SwiGLU, 5 bias, 6
bias + GELU; tiles 0-10 the ring kernel's, from 11 on the K-splitting one's."""

from __future__ import annotations

import pytest

import random

import pytest

from ppu_amd import _lib

# per kind and tile of the default plan a shape that takes it, ragged in tokens
# and columns: (tokens, columns, stages of 128 bytes of K); the K-splitting
# tiles (from 11 on) with few pieces of K and, tile for tile, with many
_DIRECT = {2: (401, 8317, 3), 3: (770, 5117, 5), 5: (770, 8317, 3), 6: (129, 8317, 3), 8: (333, 4301, 3),
           10: (6001, 1999, 16), 11: (31, 300, 3), 12: (31, 4301, 3), 13: (15, 8317, 3), 14: (2049, 200, 3),
           15: (33, 8317, 3), 16: (20001, 30, 3), 17: (65, 8317, 3), 18: (97, 8317, 3)}
_KSPLIT = {t: s for t, s in _DIRECT.items() if t > 10}
_SWIGLU = {0: (20001, 100, 3), 9: (513, 8317, 16), 13: (31, 300, 3), 15: (33, 4301, 3), 17: (20001, 3, 3),
           20: (97, 4301, 3), 21: (15, 8317, 3)}
SHAPES = {
    0: _DIRECT, 5: _DIRECT, 6: _DIRECT,
    1: {**_SWIGLU, 3: (129, 8317, 3), 22: (97, 8317, 3)},
    2: {**_DIRECT, 8: (65, 8317, 3), 17: (257, 3456, 3), 18: (401, 3456, 3)},
    3: {**_KSPLIT, 0: (770, 8317, 3), 1: (129, 8317, 3), 2: (641, 8317, 3), 3: (401, 8317, 3),
        9: (6001, 1999, 16), 19: (600, 2500, 3), 20: (6001, 300, 3)},
    4: {**_SWIGLU, 3: (97, 8317, 3)},
}


def cases(kind):
    """(tile, tokens, columns, K) of every tile that the kind's plan may take."""
    stage = 128 if kind in (2, 3, 4) else 64
    return [(t, m, n, stage * nk) for t, (m, n, few) in sorted(SHAPES[kind].items())
            for nk in ((few, 21) if t > 10 else (few,))]


@pytest.mark.parametrize("kind", range(7))
def test_every_tile_has_a_shape(kind):
    """The shapes that the kernels are tested at run on the tiles they stand for,
    and no sampled shape runs on another."""
    plan = _lib.load().q35_gemm_plan
    assert [(plan(m, n, k, kind), m, n, k) for _, m, n, k in cases(kind)] == cases(kind)
    r, stage, seen = random.Random(kind), 128 if kind in (2, 3, 4) else 64, set()
    for _ in range(60000):
        seen.add(plan(int(2 ** r.uniform(0, 17)), int(2 ** r.uniform(0, 15)), stage * int(2 ** r.uniform(0, 7.6)), kind))
    assert seen <= set(SHAPES[kind])


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
