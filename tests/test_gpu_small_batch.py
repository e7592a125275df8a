"""Small-batch mul_mat (2 .. 64 activation rows, small_batch.hip) through the
GGML boundary, every format against the oracle: the edges of its 16-row and
16-token tiles, partial 256-value units, rows at every record alignment, the
quantized src1, and the launch that ran."""
import numpy as np
import pytest

import oracle as o
from .test_gpu_ggml import FMTS, TYPE, make_weights, run, run_id

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
    # 2 and 5 units over 4 .. 8 waves, a partial weight tile (4 rows: the shortest
    # values of one GEMV pass that the kernel takes)
    names = launched(hip, fmt, 4096 if m == 4 else 512 if m % 2 else 1280, 75, m)
    assert "small_mfma_gemm" in names, names


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("n,units", [(1, 1), (16, 3), (17, 17), (530, 33)])
def test_weight_tiles_and_long_rows(hip, fmt, n, units):
    run(hip, fmt, 256 * units, n, 5)


@pytest.mark.parametrize("fmt,first", [("q4_k", 2), ("q5_k", 2), ("q4_0", 3), ("mxfp4", 4), ("nvfp4", 4)])
def test_fewest_rows(hip, fmt, first):
    assert "small_mfma_gemm" in launched(hip, fmt, 4096, 4096, first)
    assert not any("gemm" in name for name in launched(hip, fmt, 4096, 4096, first - 1))


@pytest.mark.parametrize("fmt,m,k,n,small", [
    ("q4_0", 3, 1024, 64, False), ("q5_k", 2, 1024, 64, False), ("q6_k", 4, 2048, 64, False),
    ("iq2_xs", 4, 256, 40, False), ("q4_1", 4, 3840, 64, False), ("q4_1", 4, 4096, 64, True),
    ("q4_0", 3, 1024, 8191, False), ("q4_0", 3, 1024, 8192, True),
    ("q5_k", 4, 1024, 4096, True), ("q5_k", 4, 1024, 4095, False), ("q4_1", 4, 1024, 4096, False),
    ("q4_k", 2, 256, 16, True), ("q4_0", 5, 256, 16, True),
])
def test_one_gemv_pass(hip, fmt, m, k, n, small):
    """A short batch of one GEMV pass stays one launch; more rows, and Q4_K's
    longer pass, take the kernel, as does a quantized src1."""
    assert ("small_mfma_gemm" in launched(hip, fmt, k, n, m)) == small
    if m >= 4:
        assert launched(hip, fmt, k, n, m, prequant=True) == ["small_mfma_gemm"]


@pytest.mark.parametrize("fmt,m,k,n,small", [
    ("q4_k", 32, 512, 4096, True), ("q4_k", 32, 512, 4097, False), ("q4_k", 17, 768, 8192, True),
    ("q4_k", 17, 768, 8193, False),
    ("q4_k", 33, 256, 6144, True), ("q4_k", 33, 256, 6145, False), ("q4_k", 16, 256, 13108, True),
    ("q4_k", 16, 256, 13109, False), ("mxfp4", 20, 256, 14000, True), ("mxfp4", 20, 256, 14001, False),
    ("mxfp4", 20, 3328, 12288, True), ("mxfp4", 20, 3328, 12289, False),
])
def test_most_rows(hip, fmt, m, k, n, small):
    """Both sides of the limits to the prefill GEMM (weights of zeros: which
    kernel runs, and zeros out)."""
    from weft_amd import _lib, ggml as G
    w = hip.torch.zeros(n * o.record_bytes(fmt, k), dtype=hip.torch.uint8, device=hip.dev)
    x, y = hip.empty(4 * m * k), hip.empty(4 * m * n, fill=0xA5)
    s0, s1 = G.tensor(TYPE[fmt], (k, n), w.data_ptr()), G.tensor(G.F32, (k, m), x.ptr)
    work = hip.empty(G.mul_mat_work_size(s0, s1))
    _lib.launch_log()
    G.mul_mat(s0, s1, G.tensor(G.F32, (n, m), y.ptr), work.ptr, work.nbytes)
    hip.torch.cuda.synchronize()
    assert ("small_mfma_gemm" in _lib.launch_log()) == small
    assert not y.numpy(np.float32).any()


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


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("m", [5, 20])
def test_values_that_are_not_finite(hip, fmt, m):
    """Activations and weight scales at and past the ends of fp16: outputs are
    NaN, inf (and of which sign) and finite where GGML's are, the finite ones
    within the usual bound.  (Q4_K, Q5_K and Q6_K, whose superblocks GGML sums in
    eight parts, so that an infinite scale gives infinities of both signs: finite
    where GGML's are.)"""
    from weft_amd import _lib, ggml as G
    n, k = 48, 768
    rng = np.random.default_rng(31)
    w = make_weights(fmt, n, k, 5).copy()
    x = o.seeded_normal(6, (m, k))
    act = o.ACT_OF[fmt]
    if act == "q8_k":
        x[1, 256:512] *= 1e20
    else:
        x[1, 64:96] *= 1e8      # the block's fp16 scale is inf
        x[2, 64:96] = 0.0
        x[2, 65] = 1e8          # ... with one value that is not 0
        x[3] = 0.0              # an all-zero token
    if fmt != "mxfp4" and fmt != "nvfp4":
        elems, nbytes = (256, o.record_bytes(fmt, 256)) if act == "q8_k" else (32, o.record_bytes(fmt, 32))
        rec = w.reshape(n, k // elems, nbytes)
        at = 208 if fmt == "q6_k" else 0
        for row, bits in ((3, 0x7C00), (4, 0xFC00), (5, 0x7BFF), (6, 0x0001), (7, 0x0000)):
            rec[row, 1, at:at + 2] = np.array([bits], np.uint16).view(np.uint8)
    else:
        for row in range(8, 12):  # rows with zero scales and zero codes
            w[row] = w[row] * (rng.random(w.shape[1]) < 0.7)
    xq = o.quantize(act, x)
    g = o.mul_mat_q(fmt, w, xq, n, k, m)
    e, a = o.mul_mat_f64(fmt, w, xq, n, k, m)
    wd, xd, yd = hip.to_dev(w), hip.to_dev(x), hip.empty(4 * n * m)
    s0, s1 = G.tensor(TYPE[fmt], (k, n), wd.ptr), G.tensor(G.F32, (k, m), xd.ptr)
    work = hip.empty(G.mul_mat_work_size(s0, s1))
    _lib.launch_log()
    G.mul_mat(s0, s1, G.tensor(G.F32, (n, m), yd.ptr), work.ptr, work.nbytes)
    hip.torch.cuda.synchronize()
    assert "small_mfma_gemm" in _lib.launch_log()
    y = yd.numpy(np.float32).reshape(m, n)
    assert (~np.isfinite(g)).any() and np.isfinite(g).any()
    np.testing.assert_array_equal(np.isfinite(y), np.isfinite(g))
    if fmt in ("q4_k", "q5_k", "q6_k"):
        y, g = np.where(np.isfinite(y), y, np.nan), np.where(np.isfinite(g), g, np.nan)
    np.testing.assert_array_equal(np.isnan(y), np.isnan(g))
    np.testing.assert_array_equal(np.where(np.isinf(y), np.sign(y), 0), np.where(np.isinf(g), np.sign(g), 0))
    fin = np.isfinite(g)
    assert o.within_tolerance(y[fin], g[fin].astype(np.float64), a[fin]).all()


@pytest.mark.parametrize("fmt", ["q4_k", "q5_k"])
@pytest.mark.parametrize("m", [3, 15])
def test_any_bsums(hip, fmt, m):
    """A Q8_K src1 whose bsums are a caller's own, up to the ends of int16 and
    not the sums of its values (which are at most 2048): they are taken as they
    are, as GGML's vec_dot does."""
    from weft_amd import ggml as G
    n, k = 40, 1024
    rng = np.random.default_rng(33)
    w = make_weights(fmt, n, k, 34)
    xq = o.quantize("q8_k", o.seeded_normal(35, (m, k))).reshape(m, k // 256, 292)
    bs = rng.integers(-32768, 32768, size=(m, k // 256, 16)).astype(np.int16)
    bs[0, 0], bs[0, 1], bs[1, 0] = -32768, 32767, 2049
    xq[:, :, 260:] = bs.view(np.uint8).reshape(m, k // 256, 32)
    xq = np.ascontiguousarray(xq.reshape(m, -1))
    want = o.mul_mat_q(fmt, w, xq, n, k, m)
    wd, xd, yd = hip.to_dev(w), hip.to_dev(xq), hip.empty(4 * n * m)
    G.mul_mat(G.tensor(TYPE[fmt], (k, n), wd.ptr), G.tensor(G.Q8_K, (k, m), xd.ptr), G.tensor(G.F32, (n, m), yd.ptr))
    hip.torch.cuda.synchronize()
    y = yd.numpy(np.float32).reshape(m, n)
    # fp32 sums of the same integers: eight roundings a superblock of GGML's 1 / 2 ulp, and this kernel's
    assert np.abs(y - want).max() <= 2e-6 * np.abs(want).max()


@pytest.mark.parametrize("fmt,n,k,m", [
    ("q4_0", 4090, 2304, 20), ("q4_0", 4112, 2304, 20),    # eight waves; 257 workgroups: four
    ("q4_0", 12288, 1024, 17), ("q4_0", 12304, 1024, 17),  # four waves; 769 workgroups: two
    ("q4_1", 8208, 1280, 33), ("q5_k", 12304, 768, 20),    # two waves, uneven shares of the units
])
def test_waves_of_a_workgroup(hip, fmt, n, k, m):
    """Each choice of the waves that share K, on both sides of where it changes."""
    assert "small_mfma_gemm" in launched(hip, fmt, k, n, m)


@pytest.mark.parametrize("fmt,n,k,experts,used,m,small", [
    ("q4_k", 10240, 4096, 4, 1, 3, False), ("q4_k", 10240, 4096, 4, 1, 4, True),
    ("q4_k", 10240, 4096, 8, 1, 5, False), ("q4_k", 10239, 4096, 8, 1, 5, True),
    ("q4_k", 10239, 4096, 4, 2, 2, False),
    ("q4_k", 8192, 4096, 4, 1, 3, False), ("q4_k", 8192, 4096, 4, 1, 4, True),
    ("q4_k", 4096, 8192, 4, 1, 2, False), ("q4_k", 4096, 8448, 4, 1, 2, True),
    ("q4_k", 6144, 4096, 3, 1, 2, False), ("q4_k", 6144, 4096, 3, 1, 3, True),
    ("q4_k", 4096, 4096, 4, 1, 2, True),
    ("q4_k", 14336, 2048, 4, 1, 2, False), ("q4_k", 28672, 1024, 4, 1, 2, True),
    ("nvfp4", 10240, 4096, 4, 1, 2, False), ("nvfp4", 10240, 4096, 4, 1, 3, True),
    ("nvfp4", 10240, 4096, 4, 2, 2, True), ("q5_k", 10240, 4096, 4, 1, 2, True),
])
def test_pairs_that_share_little(hip, fmt, n, k, experts, used, m, small):
    """Few pairs of large matrices stay on the pair GEMV (weights of zeros: which
    kernel runs, and zeros out)."""
    from weft_amd import _lib, ggml as G
    w = hip.torch.zeros(experts * n * o.record_bytes(fmt, k), dtype=hip.torch.uint8, device=hip.dev)
    x, y = hip.empty(4 * m * k), hip.empty(4 * m * used * n, fill=0xA5)
    ids = hip.to_dev(np.array([[(t + s) % experts for s in range(used)] for t in range(m)], np.int32))
    s0, s1 = G.tensor(TYPE[fmt], (k, n, experts), w.data_ptr()), G.tensor(G.F32, (k, 1, m), x.ptr)
    it = G.tensor(G.I32, (used, m), ids.ptr)
    work = hip.empty(G.mul_mat_id_work_size(s0, s1, it))
    _lib.launch_log()
    G.mul_mat_id(s0, s1, it, G.tensor(G.F32, (n, used, m), y.ptr), work.ptr, work.nbytes)
    hip.torch.cuda.synchronize()
    assert ("small_mfma_gemm_grouped" in _lib.launch_log()) == small
    assert not y.numpy(np.float32).any()


@pytest.mark.parametrize("fmt,k,pad", [("q4_k", 512, 2), ("q5_k", 512, 2), ("q6_k", 512, 1), ("iq2_xxs", 768, 0),
                                       ("iq2_xs", 768, 0)])
def test_many_q8k_rows_no_gemm_takes(hip, fmt, k, pad):
    # a Q8_K src1 on weights off 4-byte alignment (Q6_K: off 2), an odd superblock count
    assert launched(hip, fmt, k, 75, 70, pad_w=pad, prequant=True) == ["small_mfma_gemm"]
