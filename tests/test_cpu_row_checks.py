"""The host checks of the row passes and of a sequence of grouped products: what an entry point would
write out of place, or refuse half-way through, is refused before anything is enqueued."""

import numpy as np
import pytest
import torch

from apexw_amd import _lib as L


@pytest.mark.parametrize("dtype,size", [(L.F32, 4), (L.BF16, 2), (L.F16, 2)])
def test_row_stats_check_covers_both_halves(dtype, size):
    """apexw_grad_row_stats writes a mean and a sum of squares per row: an output whose second half reaches
    into the grad is refused; apexw_check_row_means still accepts what apexw_grad_row_means writes."""
    lib, rows, row_len, g = L.load(), 16, 8, 1 << 20
    prep = np.zeros(1, dtype=L.GRAD_PREP_DTYPE)
    prep["g"], prep["n"], prep["row_len"], prep["dtype"] = g, rows * row_len, row_len, dtype

    def status(out):
        prep["out"] = out
        return lib.apexw_check_row_means(prep.ctypes.data), lib.apexw_check_row_stats(prep.ctypes.data)

    end = g + rows * row_len * size
    assert status(g - 2 * rows * 4) == (0, 0) and status(end) == (0, 0)
    assert status(g - 2 * rows * 4 + 4) == (0, 1) and status(g - rows * 4) == (0, 1)
    assert status(g - rows * 4 + 4) == (1, 1) and status(end - 4) == (1, 1)
    prep["row_len"] = 7
    assert status(end) == (1, 1)
    prep["row_len"] = row_len
    assert status(end + 2) == (4, 4)
