"""The FP32 one-half product on both sides of each line of the rule that picks its
workgroups (fewer than 128, 128 to 256, 257 to 383 and more four-wave workgroups),
over 1, 2, 4 and 8 column slices: 40, 80, 160 and 320 of them at 5000 samples,
64 to 512 at 8100, 48 to 384 at 6100."""
import pytest

from test_gpu_gemm_half import test_half_product as half_product

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [5000, 6100, 8100])
def test_half_product_workgroups(session, N):
    half_product(session, N)
