"""Which gradients the kernels of a wide projection read in place: rows of pieces of eight elements that the storage holds whole (CPU: the
predicate reads strides, addresses and the storage's size)."""

import pytest
import torch

from minitrain_amd import _lib


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("start", [0, 8])
@pytest.mark.parametrize("columns", [64, 65, 71, 72])
def test_the_storage_holds_the_last_piece(columns, start, dtype):
    fits, rows, pitch = _lib.host().linear_rows_fit, 130, 72
    for behind in range(10):   # elements behind the last one that the storage holds
        storage = torch.zeros(start + (rows - 1) * pitch + columns + behind, dtype=dtype)
        assert fits(storage.as_strided((rows, columns), (pitch, 1), start)) == (columns + behind >= -(-columns // 8) * 8), behind


def test_rows_that_are_not_whole_pieces_apart_do_not_fit():
    fits, storage = _lib.host().linear_rows_fit, torch.zeros(4096, dtype=torch.bfloat16)
    assert fits(storage.as_strided((10, 16), (24, 1), 8)) and fits(storage.as_strided((10, 16), (16, 1), 0))
    for stride, start in (((23, 1), 0), ((24, 2), 0), ((24, 1), 4), ((8, 1), 0), ((0, 1), 0)):
        assert not fits(storage.as_strided((10, 16), stride, start)), (stride, start)
