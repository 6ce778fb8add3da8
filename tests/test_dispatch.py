"""Which kernel the size rules pick (CPU only): the tables are read from the sources and evaluated as the entry points do, so
that the GPU tests' labelled shapes keep reaching the kernels they are there for when the tables are fitted again."""
import re

import numpy as np
import pytest

from kern_glm53_amd import build

CUS = 256


def _shapes(source, fields):
    """The rows of the `shapes` table in a source file."""
    text = (build.CSRC / source).read_text()
    body = re.search(r"static const Shape shapes\[\] = \{(.*?)\};\n", text, re.S).group(1)
    rows = [tuple(float(x.rstrip("f")) for x in re.findall(r"[\d.]+f?", row)) for row in re.findall(r"\{([^{}]*)\}", body)]
    assert rows and all(len(r) == fields for r in rows), rows
    return rows


def dense_tile(m, n, k, ldc=None):
    """kg_fp8_gemm's pick for an A and C within the persistent kernel's reach: (rows, columns, workgroups a CU)."""
    ldc = n if ldc is None else ldc
    best = None
    for bm, bn, per_cu, fixed, block, start in _shapes("kg_fp8_gemm.hip", 6):
        if (bm, bn) == (256, 256) and (n % 8 or ldc % 8):
            continue
        tiles = -(-m // int(bm)) * -(-n // int(bn))
        rounds = np.float32(-(-tiles // (int(per_cu) * CUS)))
        us = np.float32(start) + rounds * (np.float32(fixed) + np.float32(block) * np.float32(k >> 7))
        if best is None or us < best[0]:
            best = us, (int(bm), int(bn), int(per_cu))
    return best[1]


def library_tile(m, n, k):
    """The tile of a library GEMM (kg_gemm_bf16, kg_gemm_bf16_f32) with n > 64 and k >= 1024."""
    best = None
    for b, fixed, step in _shapes("kg_bf16_batched.hip", 3):
        tiles = -(-m // int(b)) * -(-n // int(b))
        us = np.float32(-(-tiles // CUS)) * (np.float32(fixed) + np.float32(step) * np.float32(k >> 6))
        if best is None or us < best[0]:
            best = us, int(b)
    return best[1]


def batched_columns(heads, m, n):
    """The column tile of the head-batched kernel (a library GEMM below k = 1024 is one head of it)."""
    text = (build.CSRC / "kg_bf16_batched.hip").read_text()
    limit = int(re.search(r"const int bn = n >= 256 && .*>= (\d+) \? 256 : 128;", text).group(1))
    return 256 if n >= 256 and heads * -(-m // 128) * -(-n // 256) >= limit else 128


@pytest.mark.parametrize("m,n,k,ldc,tile", [
    (7, 2752, 6144, 2752, (32, 32, 1)), (150, 20480, 2048, 20480, (128, 192, 1)), (16384, 6144, 16384, 6144, (256, 256, 1)),
    (5000, 2752, 6144, 2752, (256, 256, 1)), (5000, 2752, 6144, 2756, (128, 192, 1)),
])
def test_dense_tile(m, n, k, ldc, tile):
    assert dense_tile(m, n, k, ldc) == tile


def test_gpu_dense_cases_reach_every_tile():
    """The tile-shape cases of the dense GEMM's GPU test run the tiles they are listed under."""
    from tests.test_gpu_gemm import PERSISTENT, TILE_SHAPES
    for tile, cases in TILE_SHAPES.items():
        for m, n, k in cases:
            assert dense_tile(m, n, k, (n + 3) // 4 * 4 + 4) == tile, (tile, m, n, k)
    for m, n, k, rows, lda, ldc, sfa_rows in PERSISTENT:
        assert dense_tile(m, n, k, ldc) == (256, 256, 1), (m, n, k)
    assert {0 < m % 256 <= 128 for m, *_ in PERSISTENT} == {True, False}             # half-tile tails and others


def test_gpu_library_cases_reach_every_tile():
    from tests.test_gpu_gemm import LIBRARY_128, LIBRARY_FEW, WIDE_BATCHED, WIDE_F32
    assert all(library_tile(m, n, k) == 128 for m, n, k, ldc in LIBRARY_128)
    assert {library_tile(m, n, k) for m, n, k in LIBRARY_FEW} == {32, 64}
    assert all(batched_columns(heads, m, n) == 256 and n % 256 for heads, m, n, k in WIDE_BATCHED)
    assert all(k < 1024 and batched_columns(1, m, n) == 256 and n % 256 for m, n, k, ldc in WIDE_F32)
