"""Where the middling tiles leave a product to other kernels (`kernl_linear_mid_kind`, answered on the host)."""
import pytest

from kernl_amd import _lib


# many rows against a cached weight; one row tile over a long K, plain and gated
@pytest.mark.parametrize("rows, n, k, gated", [(3204, 3072, 2560, False), (3999, 3072, 2048, False), (4082, 2304, 2560, False),
                                               (3958, 4096, 1536, False), (3369, 4096, 2048, False), (3059, 5120, 1536, False),
                                               (1777, 3072, 2048, False), (2343, 2304, 2560, False),
                                               (108, 12288, 11008, False), (89, 11008, 11008, False), (128, 10240, 11008, True)], ids=str)
def test_left_to_the_others(rows, n, k, gated):
    assert _lib.linear_mid_kind(rows, n, k, gated) == 0


# few columns, a large weight; a K of 8192 or less; many column tiles  (3810 x 2560 x 2048 and 2603 x 3072 x 2048 are level: 47.2 and 33.0 us on
# these tiles, 45.3 and 31.7 on the wide ones)
@pytest.mark.parametrize("rows, n, k, gated", [(3003, 3072, 5120, False), (3500, 768, 3072, False), (4096, 1024, 4096, False), (1300, 3072, 2048, False),
                                               (91, 11008, 8192, False), (125, 12288, 5120, True), (69, 28672, 12288, True)], ids=str)
def test_kept(rows, n, k, gated):
    assert _lib.linear_mid_kind(rows, n, k, gated) >= 11
