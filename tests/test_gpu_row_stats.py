"""GPU: the row means with the clip's row sums (apexw_grad_row_stats), and the tensor norms of
tensors with few and many partial sums, against float64 sums.

Bars: the mean is the fp32 row sum over the row length rounded to the grad dtype, so it lies within
one unit of that dtype of the float64 mean plus the fp32 sum's error; a row's sum of squares adds
row_len non-negative fp32 terms in at most row_len / 64 + 70 roundings each (a lane's share, the wave,
the ragged ends), so its relative error is below that times 2^-24.
"""

import numpy as np
import pytest
import torch

from apexw_amd import _lib as L

pytestmark = pytest.mark.gpu


def _upload(a):
    return torch.from_numpy(a.view(np.uint8).copy()).cuda()


@pytest.mark.parametrize("dtype,code", [(torch.bfloat16, L.BF16), (torch.float32, L.F32), (torch.float16, L.F16)])
@pytest.mark.parametrize("row_len", [1, 7, 511, 512, 4095, 4096, 4104, 6152, 14336])
def test_row_stats_match_float64(dtype, code, row_len):
    rows = 37
    gen = torch.Generator().manual_seed(row_len)
    g = (torch.randn(rows, row_len, generator=gen) * 1e-2 + 3e-3).to(dtype)
    g[5, row_len // 2] = float("nan")
    g[6, -1] = float("inf")
    dg = g.cuda()
    out = torch.full((2 * rows,), -1.0, device="cuda")
    prep = np.zeros(1, dtype=L.GRAD_PREP_DTYPE)
    prep["g"], prep["out"], prep["n"], prep["row_len"], prep["dtype"] = dg.data_ptr(), out.data_ptr(), g.numel(), \
        row_len, code
    assert L.load().apexw_check_row_means(prep.ctypes.data) == 0
    units = np.zeros(rows, dtype=L.UNIT_DTYPE)
    units["unit"] = np.arange(rows)
    dp, du = _upload(prep), _upload(units)
    L.check(L.load().apexw_grad_row_stats(dp.data_ptr(), 1, du.data_ptr(), rows, 1.0, L.HP_SANITIZE, None,
                                          torch.cuda.current_stream().cuda_stream), "row stats")
    got = out.cpu()
    clean = torch.nan_to_num(g, nan=0.0, posinf=65504.0, neginf=-65504.0).double()
    mean = clean.mean(dim=1)
    ulp = {torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -23, torch.float16: 2.0 ** -11}[dtype]
    err = (row_len / 64 + 70) * 2.0 ** -24
    bound = mean.abs() * ulp + err * clean.abs().mean(dim=1) + (6e-8 if dtype == torch.float16 else 1e-30)
    assert bool(((got[:rows].double() - mean).abs() <= bound).all())
    # about the mean that was stored, in the grad dtype
    diff = (clean.float() - got[:rows].unsqueeze(1)).to(dtype).double()
    want = diff.square().sum(dim=1)
    assert bool(((got[rows:].double() - want).abs() <= err * want + 1e-30).all())


@pytest.mark.parametrize("n_tensors", [3, 2100])
def test_tensor_norms_of_few_and_many_partials(n_tensors):
    """One tensor beyond 1024 units (summed by a workgroup) among small ones (a wave each), with one
    workgroup per tensor and with 16 tensors to a workgroup."""
    from apexw_amd import ApexW
    gen = torch.Generator(device="cuda").manual_seed(3)
    sizes = [64 + i % 50 for i in range(n_tensors)]
    sizes[n_tensors // 2] = 2048 * 1025 + 13
    sizes[0] = 2048 * 1024
    params = [torch.nn.Parameter(torch.zeros(n, device="cuda")) for n in sizes]
    for p in params:
        p.grad = torch.randn(p.shape, device="cuda", generator=gen)
    opt = ApexW(params, lr=1e-3, clip_grad_norm=0.5)
    opt.step()
    coef = float(next(iter(opt._plans.values())).clip_ws[2])
    total = sum(float(p.grad.double().square().sum()) for p in params) ** 0.5
    # the fp32 partial sums of each unit and of the norms: far below 1e-5 relative
    assert abs(coef - 0.5 / (total + 1e-6)) <= 1e-5 * coef
