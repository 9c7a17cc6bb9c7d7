"""Which products leave K whole (`kernl_linear_split_workspace_bytes`, answered on the host)."""
import pytest

from kernl_amd import _lib

STATS, NORM = _lib.FINISH_RMS_STATS, _lib.FINISH_LAYER_NORM


# wide products of few rows, in one pass over K on 64 x 32 tiles
@pytest.mark.parametrize("rows, n, k, finish", [(67, 4096, 2048, NORM), (178, 2048, 1536, NORM), (265, 1536, 2048, NORM)], ids=str)
def test_one_pass(rows, n, k, finish):
    assert _lib.linear_split_workspace_bytes(rows, n, k, finish) == 0


# narrow products over a long K, and statistics to come
@pytest.mark.parametrize("rows, n, k, finish", [(207, 2048, 3072, STATS), (1000, 768, 3072, STATS), (231, 768, 3072, STATS), (231, 768, 3072, NORM),
                                               (500, 768, 3072, STATS), (500, 768, 3072, NORM),
                                               (333, 4096, 4096, STATS), (333, 4096, 11008, STATS), (2079, 1024, 11008, NORM)], ids=str)
def test_split(rows, n, k, finish):
    assert _lib.linear_split_workspace_bytes(rows, n, k, finish) > 0
