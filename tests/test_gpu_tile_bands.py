"""Prefill GEMMs on more than eight 64-token tiles, whose tiles are walked in
bands (nine tiles: 5 + 4, eighteen: 6 + 6 + 6, nineteen with a last one of one
row), and Q6_K rows on both sides of its four-superblock partial sums; against
the oracle."""
import pytest

from .test_gpu_ggml import run

pytestmark = pytest.mark.gpu

FORMATS = ["q4_0", "q4_1", "mxfp4", "nvfp4", "q4_k", "q5_k", "q6_k", "iq2_xxs", "iq2_xs"]


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("m,n", [(513, 300), (1152, 129), (1153, 40)])
def test_bands(hip, fmt, m, n):
    run(hip, fmt, 256, n, m)


@pytest.mark.parametrize("superblocks", [3, 4, 5, 8, 9])
def test_q6k_partial_sums(hip, superblocks):
    run(hip, "q6_k", 256 * superblocks, 130, 65)
