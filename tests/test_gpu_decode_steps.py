"""Batch-1 GEMVs with the records in registers on rows longer than one step of
4096 values (their waves split a row into up to four steps), and Q6_K rows
that are only 2-byte aligned; against the oracle, with the kernel that ran."""
import pytest

from .test_gpu_ggml import run

pytestmark = pytest.mark.gpu

KERNEL = {"q4_0": "rec_gemv_m1_kernel", "q4_1": "rec_gemv_m1_kernel", "mxfp4": "rec_gemv_m1_kernel",
          "nvfp4": "rec_gemv_m1_kernel", "q5_k": "q5k_gemv_m1_kernel", "q6_k": "q6k_gemv_m1_kernel"}


def launched(hip, *args, **kwargs):
    from weft_amd import _lib
    _lib.launch_log()
    run(hip, *args, **kwargs)
    return _lib.launch_log()


@pytest.mark.parametrize("fmt", list(KERNEL))
@pytest.mark.parametrize("k,n", [
    (4352, 300), (8192, 17), (8448, 5),     # two steps (uneven, full), three with short steps
    (11008, 1100), (12288, 1), (16384, 40),  # three steps over many rows, one row, four full steps
])
def test_steps(hip, fmt, k, n):
    assert launched(hip, fmt, k, n, 1) == [KERNEL[fmt]]


@pytest.mark.parametrize("fmt,k", [("q4_0", 4160), ("q4_1", 12352), ("mxfp4", 4224), ("nvfp4", 8256)])
def test_steps_of_partial_units(hip, fmt, k):
    # whole lanes of 64 values, not whole 256-value units (and rows of whole dwords)
    assert launched(hip, fmt, k, 33, 1) == [KERNEL[fmt]]


@pytest.mark.parametrize("fmt", list(KERNEL))
def test_past_four_steps(hip, fmt):
    assert launched(hip, fmt, 16640, 9, 1) == ["staged_gemv_kernel"]


@pytest.mark.parametrize("k,pad", [(256, 0), (2816, 0), (1024, 2), (4096, 6), (11008, 4)])
def test_q6k_two_byte_rows(hip, k, pad):
    assert launched(hip, "q6_k", k, 70, 1, pad_w=pad) == [KERNEL["q6_k"]]


@pytest.mark.parametrize("n,k,kernel", [(14336, 12288, "staged_gemv_kernel"), (14335, 12288, KERNEL["q6_k"]),
                                        (14336, 12032, KERNEL["q6_k"]), (14336, 12544, KERNEL["q6_k"])])
def test_q6k_many_long_rows(hip, n, k, kernel):
    """Many rows of three whole steps are the staged GEMV's (weights of zeros:
    which kernel runs, and zeros out)."""
    from weft_amd import _lib, ggml as G
    w, x = hip.torch.zeros(n * k // 256 * 210, dtype=hip.torch.uint8, device=hip.dev), hip.empty(4 * k)
    y, work = hip.empty(4 * n, fill=0xA5), hip.empty(k // 256 * 292)
    _lib.launch_log()
    G.mul_mat(G.tensor(G.Q6_K, (k, n), w.data_ptr()), G.tensor(G.F32, (k, 1), x.ptr),
              G.tensor(G.F32, (n, 1), y.ptr), work.ptr, work.nbytes)
    hip.torch.cuda.synchronize()
    assert _lib.launch_log() == [kernel]
    assert not y.numpy("float32").any()
