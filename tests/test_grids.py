"""What a launch would not hold is refused by the entries' own checks, before the launch (these need no GPU)."""
import pytest

from herbert_rs_amd.errors import BackendError
from herbert_rs_amd.kernels import lib


def grouped(M, groups, N):
    """One call of hb_grouped_mfma with nothing behind its pointers: for calls that are refused."""
    lib.call("moe", "hb_grouped_mfma", None, 32, 0, None, N, 32, None, N, 0, 0, None, 0, None, None, None, 0, M, groups,
             0.0, 0.0, 1.0, 0, None)


@pytest.mark.parametrize("M, groups, N", [(64, 65535, 256 * 256), (64, 65536, 16), (64 * 32000, 2, 600 * 256)])
def test_a_grouped_product_whose_tiles_exceed_the_grid_is_refused(M, groups, N):
    with pytest.raises(BackendError, match="exceed the grid"):
        grouped(M, groups, N)


@pytest.mark.parametrize("M, N, text", [(4194241, 16, "at most 4194240 rows"), (4194240, 1 << 20, "exceed the grid")])
def test_a_product_beyond_the_rows_or_the_grid_is_refused(M, N, text):
    with pytest.raises(BackendError, match=text):
        lib.call("gemm_plain", "hb_gemm_plain", None, 0, None, 0, None, 0, M, N, 1, 1, 1, N, 0, None)
