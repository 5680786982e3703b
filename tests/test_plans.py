"""The plans that the GPU tests of the GEMMs' tiles, K splits and walks are written for, asked of the library
without a GPU: a change of a cost model's constants that takes a test off its path fails here."""
import pytest

import test_gpu_gemm as gemms


@pytest.mark.parametrize("m,k,n,resid,tiles", gemms.PLANNED + gemms.MID_SIZES)
def test_bf16_plans(m, k, n, resid, tiles):
    assert gemms.gemm_plan(m, k, n) == tiles


@pytest.mark.parametrize("m,k,n", gemms.WALKS)
def test_bf16_walks(m, k, n):
    assert gemms.gemm_plan(m, k, n) == (256, 256, 1) and -(-m // 256) * -(-n // 256) >= 2 * 256


@pytest.mark.parametrize("m,k,inter,tile", gemms.SWIGLU_TILES)
def test_swiglu_plans(m, k, inter, tile):
    assert gemms.gemm_plan(m, k, 2 * inter, split=0) == (*tile, 1)
    assert (gemms.gemm_plan(m, k, 2 * inter)[2] > 1) == (k > 1024)


@pytest.mark.parametrize("m,k,n,tiles", gemms.FP8_PLANNED)
def test_fp8_plans(m, k, n, tiles):
    assert gemms.fp8_plan(m, k, n) == tiles


def test_every_form_is_reached():
    """Each tile of the bf16 GEMM that splits K, and each form of the fp8 GEMM."""
    split = {t[:2] for *_, t in gemms.PLANNED if t[2] > 1}
    assert split == {(256, 256), (256, 128), (128, 256), (128, 128), (64, 128)}
    assert {(t[:2], t[2] > 1) for *_, t in gemms.FP8_PLANNED} >= {
        ((r, c), s) for r, c in [(256, 256), (256, 128), (128, 128), (64, 128)] for s in (False, True)}
