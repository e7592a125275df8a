"""Small-batch mul_mat (2 .. 64 activation rows, small_batch.hip) through the
GGML boundary, every format against the oracle: the edges of its 16-row and
16-token tiles, partial 256-value units, rows at every record alignment, the
quantized src1, and the launch that ran."""
import numpy as np
import pytest

import oracle as o
from .test_gpu_ggml import FMTS, run, run_id

pytestmark = pytest.mark.gpu

ELEMS = {"q4_0": 32, "q4_1": 32, "mxfp4": 32, "nvfp4": 64}


def launched(hip, *args, **kwargs):
    from weft_amd import _lib
    _lib.launch_log()
    run(hip, *args, **kwargs)
    return _lib.launch_log()


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("m", [4, 15, 16, 17, 32, 33, 64])
def test_token_tiles(hip, fmt, m):
    # 2 and 5 units over 4 .. 8 waves, a partial weight tile
    names = launched(hip, fmt, 512 if m % 2 else 1280, 75, m)
    assert "small_mfma_gemm" in names, names


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("n,units", [(1, 1), (16, 3), (17, 17), (530, 33)])
def test_weight_tiles_and_long_rows(hip, fmt, n, units):
    run(hip, fmt, 256 * units, n, 5)


@pytest.mark.parametrize("fmt,first", [("q4_k", 2), ("q5_k", 2), ("q4_0", 3), ("mxfp4", 4), ("nvfp4", 4)])
def test_fewest_rows(hip, fmt, first):
    assert "small_mfma_gemm" in launched(hip, fmt, 512, 64, first)
    assert not any("gemm" in name for name in launched(hip, fmt, 512, 64, first - 1))


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("m", [16, 40])
def test_bound_tiles_keep_the_prefill_gemm(hip, fmt, m):
    """A bound tile (weft_hip_set_tile_binding) keeps a small batch on the
    kernels the binding shapes: the prefill GEMM at its smallest sizes."""
    from weft_amd import _lib
    lib = _lib.load()
    try:
        assert lib.weft_hip_set_tile_binding(b"MC", 64) == 1
        names = launched(hip, fmt, 512, 75, m)
    finally:
        lib.weft_hip_clear_tile_bindings()
    assert any("gemm" in n and not n.startswith("small") for n in names), names


@pytest.mark.parametrize("fmt", list(ELEMS))
@pytest.mark.parametrize("records", [1, 7, 9])
def test_partial_units(hip, fmt, records):
    # rows that are not whole 256-value units
    run(hip, fmt, ELEMS[fmt] * records, 40, 5)


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("pad", [1, 3, 5])
def test_row_alignment(hip, fmt, pad):
    # each record alignment: rows start at every offset of a 16-byte chunk
    run(hip, fmt, 768, 35, 9, pad_w=pad if fmt in ("mxfp4", "q6_k", "nvfp4") else 2 * pad, pad_x=1, pad_y=3)


@pytest.mark.parametrize("fmt", FMTS)
def test_quantized_src1(hip, fmt):
    names = launched(hip, fmt, 768, 50, 21, prequant=True)
    assert names == ["small_mfma_gemm"], names


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("ne11", [1, 2])
def test_mul_mat_id_pairs(hip, fmt, ne11):
    """A few pairs grouped in the kernel: 19 pairs of one expert (two tiles of
    16), one token with the same expert twice, invalid ids left untouched."""
    from weft_amd import _lib
    ids = np.random.default_rng(6).integers(0, 5, size=(14, 2))
    ids[:9] = 3
    ids[10] = (-1, 5)
    _lib.launch_log()
    run_id(hip, fmt, 768, 50, 5, 2, ne11, 14, ids, pad_w=1 if fmt in ("mxfp4", "q6_k", "nvfp4") else 2)
    assert "small_mfma_gemm_grouped" in _lib.launch_log()


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("pad", [0, 1])
def test_many_rows_no_gemm_takes(hip, fmt, pad):
    """More rows than a small batch where the prefill GEMM does not take the
    weights: rows off 4-byte alignment (pad), an odd superblock count (IQ2)."""
    pad_w = 0 if not pad else 1 if fmt in ("mxfp4", "q6_k", "nvfp4") else 2
    names = launched(hip, fmt, 768, 75, 70, pad_w=pad_w, pad_y=1)
    if pad_w or fmt.startswith("iq2"):
        assert "small_mfma_gemm" in names, names


@pytest.mark.parametrize("fmt", ["q4_0", "q4_1", "mxfp4", "nvfp4"])
def test_many_quantized_rows(hip, fmt):
    # a Q8_0 / Q8_1 src1, which those formats' GEMMs do not read
    assert launched(hip, fmt, 512, 75, 70, prequant=True) == ["small_mfma_gemm"]
