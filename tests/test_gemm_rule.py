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


@pytest.mark.parametrize("kind,O,K,M,form", [
    # 2^20 outputs, 576 rows, 2^19 outputs
    (Q6K, 768, 4096, 682, FEW), (Q6K, 768, 4096, 683, HALVES), (Q4K, 520, 2048, 1008, FEW), (Q4K, 520, 2048, 1009, HALVES), (Q6K, 1024, 2048, 576, FEW), (Q4K, 1536, 4096, 576, FEW),
    (Q4K, 1536, 4096, 577, HALVES), (Q4K, 2048, 4096, 512, FEW), (Q4K, 2048, 4096, 513, HALVES), (Q4K, 2560, 2048, 409, FEW), (Q4K, 2560, 2048, 410, THIN),
    (Q6K, 4088, 512, 256, FEW), (Q4K, 4096, 2048, 128, FEW), (Q4K, 4096, 2048, 129, HALVES), (Q6K, 4096, 2048, 192, FEW), (Q6K, 4096, 2048, 193, HALVES),
    # narrow ones; few slabs
    (Q4K, 512, 2048, 1536, FEW), (Q6K, 512, 2048, 1024, FEW), (Q6K, 512, 2048, 1025, THIN), (Q6K, 256, 2048, 2560, FEW), (Q4K, 2048, 512, 1024, FEW),
    (Q4K, 2048, 512, 1025, THIN), (Q4K, 2048, 1536, 2000, THIN), (Q4K, 512, 1024, 1024, FEW),
    # what the few-row kernels don't take (K, the scales' pieces)
    (Q4K, 768, 4352, 128, LDS), (Q4K, 768, 4352, 129, THIN), (Q6K, 131, 512, 129, THIN), (Q6K, 2051, 4608, 129, HALVES)])
def test_rows_at_which_the_forms_change(orn, kind, O, K, M, form):
    assert orn.gemm_form(kind, O, K, M) == form


@pytest.mark.parametrize("kind", [Q4K, Q6K])
@pytest.mark.parametrize("O,K,M,form", [
    # few full tiles: small ones up to one a compute unit (of K = 512 two), as many as 128 x 128 outputs each make
    (2560, 2048, 420, THIN), (6144, 4096, 600, THIN), (8192, 2048, 512, THIN), (8192, 2048, 513, OWN), (8192, 512, 1024, THIN), (8192, 512, 1025, OWN),
    (12288, 2048, 257, OWN)])
def test_a_launch_of_few_full_tiles_takes_small_ones(orn, kind, O, K, M, form):
    assert orn.gemm_form(kind, O, K, M) == form


@pytest.mark.parametrize("kind", [Q4K, Q6K])
@pytest.mark.parametrize("E,O,K,avg,form", [
    # what the few-row kernels don't take, from 48 pairs an expert: not of few slabs
    (16, 131, 512, 48, LDS), (256, 2048, 256, 79, LDS), (256, 512, 4352, 47, LDS), (256, 512, 4352, 48, OWN), (16, 512, 4352, 48, THIN),
    # 80 pairs an expert and more: small tiles while large ones are half the compute units or fewer
    (256, 2048, 512, 79, FEW), (256, 2048, 512, 80, OWN), (16, 2048, 512, 256, THIN), (16, 2048, 512, 257, OWN), (17, 2048, 512, 80, OWN),
    (64, 512, 2048, 207, THIN), (65, 512, 2048, 207, OWN), (16, 131, 512, 600, THIN)])
def test_experts_of_few_full_tiles_take_small_ones(orn, kind, E, O, K, avg, form):
    assert orn.gather_form(kind, E, O, K, E * avg) == form
