"""Operands seen as rows: what the checks in front of a launch say about them, without making the view or the copy."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from kernl_amd.implementations.deferred_norm import row_stride, rows_of


class _Recorder(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.calls = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.calls.append(str(func))
        return func(*args, **(kwargs or {}))


def _layouts():
    base = torch.zeros((6, 5, 4, 64), dtype=torch.float16)
    flat = torch.zeros((30 * 4 * 80 + 8,), dtype=torch.float16)
    return {
        "rows": base[0, 0], "three": base[0], "four": base, "transposed": base.transpose(1, 2), "middle": base[:, ::2], "outer": base[::3],
        "features": base[..., :32], "odd features": base[..., :36], "odd copied": base[..., :36].transpose(0, 1), "columns": base[0].transpose(1, 2),
        "flipped rows": base[0, 0].t(), "expanded": base[:1, :1, :1].expand(3, 5, 4, 64), "one row each": base[:, :1, :1], "one": base[:1, :1, :1],
        "odd rows": flat[: 30 * 4 * 76].view(30, 4, 76)[..., :64], "offset": flat[4: 4 + 30 * 64].view(3, 10, 64),
        "one odd row": flat[:68].view(1, 68)[:, :64], "one odd row of three": flat[:68].view(1, 1, 68)[..., :64], "one row, odd features": flat[:36].view(1, 1, 36),
        "wide rows": flat[: 30 * 4 * 80].view(30, 4, 80)[..., :64], "leading ones": flat[:1920].view(30, 64)[None, None],
    }


@pytest.mark.parametrize("name", list(_layouts()))
def test_it_says_what_the_rows_are(name):
    t = _layouts()[name]
    with _Recorder() as made:
        said = row_stride(t)
    assert made.calls == []
    rows = rows_of(t)
    taken = rows.stride(-1) == 1 and rows.stride(0) % 8 == 0 and rows.data_ptr() % 16 == 0
    assert (said is not None) == taken
    if taken:
        assert said == rows.stride(0)


@pytest.mark.gpu
def test_nothing_is_copied_to_look_at_the_operands():
    from kernl_amd import _lib
    from kernl_amd.implementations.split_linear import split_finish_bytes

    x = torch.randn((77, 3, 3072), device="cuda").half().transpose(0, 1)
    residual = torch.randn((77, 3, 768), device="cuda").half().transpose(0, 1)
    w = torch.randn((768, 3072), device="cuda").half()
    before = torch.cuda.memory_stats()["allocation.all.allocated"]
    assert split_finish_bytes(x, w, None, residual, _lib.FINISH_RMS_STATS) > 0
    assert torch.cuda.memory_stats()["allocation.all.allocated"] == before
