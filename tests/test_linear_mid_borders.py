"""Where the middling tiles leave a product to other kernels (`kernl_linear_mid_kind`, answered on the host)."""
import pytest

from kernl_amd import _lib


# more than 3000 rows against a cached weight of whole 192-column tiles; one row tile over a long K, plain and gated
@pytest.mark.parametrize("rows, n, k, gated", [(3204, 3072, 2560, False), (3999, 3072, 2048, False), (4082, 2304, 2560, False),
                                               (108, 12288, 11008, False), (89, 11008, 11008, False), (128, 10240, 11008, True)], ids=str)
def test_left_to_the_others(rows, n, k, gated):
    assert _lib.linear_mid_kind(rows, n, k, gated) == 0


# a ragged last column tile, up to 3000 rows, a large weight; a K of 8192 or less; many column tiles
@pytest.mark.parametrize("rows, n, k, gated", [(3810, 2560, 2048, False), (2603, 3072, 2048, False), (3003, 3072, 5120, False), (3500, 768, 3072, False),
                                               (91, 11008, 8192, False), (125, 12288, 5120, True), (69, 28672, 12288, True)], ids=str)
def test_kept(rows, n, k, gated):
    assert _lib.linear_mid_kind(rows, n, k, gated) >= 11
