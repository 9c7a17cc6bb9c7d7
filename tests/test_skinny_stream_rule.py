"""Which single-query calls read their keys and values past the memory-side cache."""
import pytest
import torch

from kernl_amd.debugger import index_lib


def _streams(keys, values):
    return index_lib().skinny_streams(tuple(keys.shape), keys.stride(), values.stride())


@pytest.mark.parametrize("head", [64, 128])
def test_storage_decides_and_not_the_shape(head):
    B, H, N = 24, 32, 3001
    whole = torch.empty((B, H, N, head), device="meta", dtype=torch.float16)
    one_head = torch.empty((B, 1, N, head), device="meta", dtype=torch.float16).expand(B, H, N, head)  # read again by every query head
    one_prefix = torch.empty((1, H, N, head), device="meta", dtype=torch.float16).expand(B, H, N, head)
    interleaved = torch.empty((B, N, H, head), device="meta", dtype=torch.float16).transpose(1, 2)
    assert _streams(whole, whole) and _streams(interleaved, whole)
    for shared in (one_head, one_prefix):
        assert not _streams(shared, shared) and not _streams(whole, shared) and not _streams(shared, whole)


def test_the_border_is_the_size_of_the_cache():
    for n, beyond in ((2048, False), (2049, True)):  # 8 x 32 x 2048 x 128 keys and as many values: 256 MB
        kv = torch.empty((8, 32, n, 128), device="meta", dtype=torch.bfloat16)
        assert _streams(kv, kv) == beyond
    # dimensions of size one carry any stride
    kv = torch.empty((1, 64, 20000, 128), device="meta", dtype=torch.float16).as_strided((1, 64, 20000, 128), (0, 20000 * 128, 128, 1))
    assert _streams(kv, kv)
