"""Q6_K prefill GEMM on weight rows that are only 2-byte aligned (an odd number
of 210-byte records a row, a 2-byte offset or row pad), dense and grouped
(MUL_MAT_ID), against the oracle, and extreme scales: its weight operands are
two int8 digits of scale x value, up to 128 x 32."""
import numpy as np
import pytest

import oracle as o
from weft_amd import ggml as G
from .test_gpu_ggml import run, run_id

pytestmark = pytest.mark.gpu


def launched(call):
    from weft_amd import _lib
    _lib.launch_log()
    call()
    return _lib.launch_log()


@pytest.mark.parametrize("superblocks,n,m,pad", [
    (1, 130, 65, 0), (3, 300, 80, 0), (43, 75, 129, 0),  # odd superblock counts, ragged tiles
    (2, 130, 65, 2), (4, 64, 70, 6),                     # whole pairs, rows 2 bytes off
])
def test_two_byte_rows(hip, superblocks, n, m, pad):
    names = launched(lambda: run(hip, "q6_k", 256 * superblocks, n, m, pad_w=pad, pad_x=4, pad_y=4))
    assert "q6k_mfma_gemm" in names, names


@pytest.mark.parametrize("superblocks,pad", [(3, 0), (2, 2), (2, 4)])
def test_two_byte_rows_grouped(hip, superblocks, pad):
    ids = np.random.default_rng(9).integers(0, 5, size=(60, 2))
    names = launched(lambda: run_id(hip, "q6_k", 256 * superblocks, 150, 5, 2, 1, 60, ids, pad_w=pad))
    assert "q6k_mfma_gemm" in names, names


@pytest.mark.parametrize("superblocks", [1, 2, 5])
def test_extreme_scales(hip, superblocks):
    """Every 16-group scale at -128, -127, 127 or 0 and values at both ends of
    the 6-bit range against activations of +-127."""
    rng = np.random.default_rng(12)
    n, k, m = 96, 256 * superblocks, 70
    w = o.random_records("q6_k", n, k, seed=13).reshape(n, superblocks, 210)
    w[:, :, :192] = rng.choice(np.array([0, 255], np.uint8), size=(n, superblocks, 192))
    w[:, :, 192:208] = rng.choice(np.array([128, 129, 127, 0], np.uint8), size=(n, superblocks, 16))
    w[:, :, 208:210] = np.full((n, superblocks, 1), 3e-4, np.float16).view(np.uint8)
    w = np.ascontiguousarray(w.reshape(n, -1))
    x = rng.choice(np.array([-1.0, 1.0, 0.5], np.float32), size=(m, k)).astype(np.float32)
    xq = o.quantize("q8_k", x)
    e, a = o.mul_mat_f64("q6_k", w, xq, n, k, m)
    wd, xd, yd = hip.to_dev(w), hip.to_dev(x), hip.empty(4 * n * m)
    s0, s1 = G.tensor(G.Q6_K, (k, n), wd.ptr), G.tensor(G.F32, (k, m), xd.ptr)
    work = hip.empty(G.mul_mat_work_size(s0, s1))
    G.mul_mat(s0, s1, G.tensor(G.F32, (n, m), yd.ptr), work.ptr, work.nbytes)
    hip.torch.cuda.synchronize()
    assert o.within_tolerance(yd.numpy(np.float32).reshape(m, n), e, a).all()


def surrounded(hip, w, offset, fill):
    """w on the GPU `offset` bytes past a 256-byte boundary, bytes `fill` around it."""
    raw = np.full(w.nbytes + 512, fill, np.uint8)
    raw[256 + offset:256 + offset + w.nbytes] = w.reshape(-1)
    t = hip.torch.from_numpy(raw).to(hip.dev)
    return t, t.data_ptr() + 256 + offset


@pytest.mark.parametrize("offset", [0, 2])
@pytest.mark.parametrize("n,k", [(1, 256), (3, 768), (33, 2816), (5, 11008), (4, 4096)])
def test_batch1_reads_the_weights_alone(hip, n, k, offset):
    """An odd number of records ends in the middle of a dword, and weights at
    an address of 2 mod 4 begin in one.  The register kernel reads whole dwords
    from a row's first one on, so it takes 4-byte aligned weights only; what lies
    around the weights changes no bit of the result."""
    from weft_amd import _lib
    w, x = o.quantize("q6_k", o.seeded_normal(21, (n, k), 0.02)), o.seeded_normal(22, (1, k))
    outs = []
    for fill in (0x00, 0xFF):
        keep, ptr = surrounded(hip, w, offset, fill)
        xq, y = hip.empty(o.record_bytes("q8_k", k)), hip.empty(4 * n)
        _lib.launch_log()
        hip.call("production_mul_mat_q6_k_decode", ptr, hip.to_dev(x), xq, y, n, k, 1)
        assert _lib.launch_log() == ["staged_gemv_kernel" if offset else "q6k_gemv_m1_kernel"]
        outs.append(y.numpy(np.float32))
    e, a = o.mul_mat_f64("q6_k", w, o.quantize("q8_k", x), n, k, 1)
    assert o.within_tolerance(outs[0].reshape(1, n), e, a).all()
    np.testing.assert_array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))


@pytest.mark.parametrize("offset", [0, 2])
@pytest.mark.parametrize("n,superblocks", [(33, 3), (129, 1), (5, 43)])
def test_prefill_reads_the_weights_alone(hip, n, superblocks, offset):
    """The GEMM's 2-byte rows, as the batch-1 kernel's: 4-byte aligned weights
    only, and what lies around them changes no bit."""
    from weft_amd import _lib
    k, m = 256 * superblocks, 70
    w, x = o.quantize("q6_k", o.seeded_normal(23, (n, k), 0.02)), o.seeded_normal(24, (m, k))
    outs = []
    for fill in (0x00, 0xFF):
        keep, ptr = surrounded(hip, w, offset, fill)
        xq, y = hip.empty(m * o.record_bytes("q8_k", k)), hip.empty(4 * m * n)
        _lib.launch_log()
        hip.call("production_mul_mat_q6_k", ptr, hip.to_dev(x), xq, y, n, k, m)
        assert _lib.launch_log()[-1] == ("small_mfma_gemm" if offset else "q6k_mfma_gemm")
        outs.append(y.numpy(np.float32).reshape(m, n))
    e, a = o.mul_mat_f64("q6_k", w, o.quantize("q8_k", x), n, k, m)
    assert o.within_tolerance(outs[0], e, a).all()
    np.testing.assert_array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
