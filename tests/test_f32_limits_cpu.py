"""What the 32-bit matrix-core kernels (csrc/f32.hip) leave to the plain ones, as the host decides it."""
import pytest

from dinfer_amd.kernels import lib


@pytest.mark.parametrize("K,taken", [(0, False), (4, True), (1022, False), (2 ** 31 - 4, False), (2 ** 31 - 68, False), (2 ** 31 - 512, False),
                                     (2 ** 31 - 516, True)])
def test_products_whose_offsets_fit(K, taken):
    """Steps of 64 k are fetched two ahead, in 32-bit numbers: k must end two segments before those do."""
    fn = lib.get("dinfer_gemm_f32_supports")
    assert bool(fn(4096, max(K, 4), 8192, max(K, 4), K)) == taken
