"""Prefill GEMMs on more than eight 64-token tiles, whose tiles are walked in
bands (nine tiles: 5 + 4, eighteen: 6 + 6 + 6, nineteen with a last one of one
row), and Q6_K rows on both sides of its four-superblock partial sums; against
the oracle.  K = 512 reaches every format's GEMM (the IQ2 ones take whole pairs
of superblocks); at 256 values they run the small-batch kernel."""
import pytest

from .test_gpu_ggml import run
from .test_gpu_parity import assert_prefill_kernel

pytestmark = pytest.mark.gpu

FORMATS = ["q4_0", "q4_1", "mxfp4", "nvfp4", "q4_k", "q5_k", "q6_k", "iq2_xxs", "iq2_xs"]


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("m,n", [(513, 300), (1152, 129), (1153, 40)])
def test_bands(hip, fmt, m, n):
    run(hip, fmt, 256, n, m)


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("m,n", [(513, 300), (1153, 40), (1601, 300)])  # 1601: 26 tiles, 8 + 8 + 8 + 2
def test_bands_on_the_gemm(hip, fmt, m, n):
    hip._lib.launch_log()
    run(hip, fmt, 512, n, m)
    assert_prefill_kernel(hip, fmt, m)


def test_q4k_walks_the_bands(hip):
    # 33 x 26 tiles, more than one a workgroup: each walks its share of them
    hip._lib.launch_log()
    run(hip, "q4_k", 512, 4200, 1601)
    assert_prefill_kernel(hip, "q4_k", 1601)


@pytest.mark.parametrize("superblocks", [3, 4, 5, 8, 9])
def test_q6k_partial_sums(hip, superblocks):
    run(hip, "q6_k", 256 * superblocks, 130, 65)
