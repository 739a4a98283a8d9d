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


def _kind_ok(kind):
    """The epilogue kinds that have a kernel: an output, no transposed one with a [k x n] B, and 128 x 128
    tiles only in panels and without a [k x n] B."""
    out = kind & (L.GEMM_OUT_C | L.GEMM_OUT_CT)
    nn, ct = kind & L.GEMM_KIND_NN, kind & L.GEMM_OUT_CT
    small, panel = kind & L.GEMM_KIND_TILE128, kind & L.GEMM_KIND_PANEL
    return bool(out) and not (nn and ct) and not (small and (nn or not panel))


@pytest.mark.skipif(torch.cuda.is_available(), reason="stand-in device pointers: run where no GPU is present")
@pytest.mark.parametrize("kind", range(-1, 66))
def test_a_sequence_with_a_bad_later_launch_enqueues_nothing(kind):
    """apexw_gemm_nt_grouped_run refuses every kind without a kernel before the first launch: with a good
    launch ahead the answer is the argument error, not the launch failure that enqueueing the first one
    gives where no GPU is present (which a sequence of good kinds does give)."""
    lib, a = L.load(), 1 << 20
    seq = np.zeros(2, dtype=L.GEMM_LAUNCH_DTYPE)
    for k in ("problems", "items", "queue_offsets"):
        seq[k] = a
    seq["n_workgroups"], seq["kind"] = L.GEMM_QUEUES, (L.GEMM_OUT_C, kind)
    ok = 0 < kind < 64 and _kind_ok(kind)
    assert lib.apexw_gemm_nt_grouped_run(seq.ctypes.data, 2, None, None) == (3 if ok else 1)
