"""The rotating product of a decode step that normalises its rows once into LDS: either end of the tokens and of K that it takes."""
import pytest

from tests.test_gpu_kernels import check_fused_qkv_rope_cache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [3, 4, 5, 8, 9, 32, 33, 49, 63])
@pytest.mark.parametrize("nq,nkv,hd,K,page", [(3, 1, 32, 72, 8), (14, 2, 64, 1024, 16), (28, 4, 128, 1032, 16), (8, 2, 128, 1016, 16), (5, 5, 48, 520, 4)])
def test_rows_normalised_once(T, nq, nkv, hd, K, page):
    check_fused_qkv_rope_cache(T, nq, nkv, hd, K, page, True)
