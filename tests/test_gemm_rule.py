"""CPU: which form of the prompt GEMM a k-quant matrix of M rows takes (host code of the library; nothing is launched)."""
import pytest

from util import Q4K, Q6K

LDS, OWN, HALVES, FEW, THIN = range(5)


@pytest.mark.parametrize("kind,O,K,M", [(Q4K, 12288, 2048, 700), (Q6K, 8192, 2048, 200), (Q4K, 2048, 4096, 700), (Q6K, 4096, 1024, 3000)])
def test_option_takes_a_matrix_off_the_own_column_form(orn, kind, O, K, M):
    """gemm_duo = 0: the rule by which matrices are gathered into launches and the one by which they run agree"""
    assert orn.gemm_form(kind, O, K, M) in (OWN, HALVES, THIN)
    try:
        orn.set_option("gemm_duo", 0)
        assert orn.gemm_form(kind, O, K, M) == LDS
    finally:
        orn.set_option("gemm_duo", 1)


@pytest.mark.parametrize("kind", [Q4K, Q6K])
@pytest.mark.parametrize("O,K,M,form", [
    # few full tiles: small ones up to one a compute unit (of K = 512 two), as many as 128 x 128 outputs each make
    (2560, 2048, 300, THIN), (6144, 4096, 600, THIN), (8192, 2048, 512, THIN), (8192, 2048, 513, OWN), (8192, 512, 1024, THIN), (8192, 512, 1025, OWN),
    (12288, 2048, 257, OWN)])
def test_a_launch_of_few_full_tiles_takes_small_ones(orn, kind, O, K, M, form):
    assert orn.gemm_form(kind, O, K, M) == form
