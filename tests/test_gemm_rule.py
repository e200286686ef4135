"""CPU: which form of the prompt GEMM a k-quant matrix of M rows takes (host code of the library; nothing is launched)."""
import pytest

from util import Q4K, Q6K

LDS, OWN, HALVES, FEW = range(4)


@pytest.mark.parametrize("kind,O,K,M", [(Q4K, 12288, 2048, 700), (Q6K, 8192, 2048, 200), (Q4K, 2048, 4096, 700), (Q6K, 4096, 1024, 3000)])
def test_option_takes_a_matrix_off_the_own_column_form(orn, kind, O, K, M):
    """gemm_duo = 0: the rule by which matrices are gathered into launches and the one by which they run agree"""
    assert orn.gemm_form(kind, O, K, M) in (OWN, HALVES)
    try:
        orn.set_option("gemm_duo", 0)
        assert orn.gemm_form(kind, O, K, M) == LDS
    finally:
        orn.set_option("gemm_duo", 1)
