"""GPU: the clip of centralized grads whose squares the row pass forms (apexw_grad_row_stats and
APEXW_HP_ROW_SUMSQ), against float64 norms and the CPU oracle's step.

Norm bars: a sum of non-negative fp32 terms in chains of at most 40 additions (a unit's 32 terms or a
row's eight running sums, the folds and the wave; partial sums meet in float64) is within 40 x 2^-24
relative, its root within half of that, and the root and its storage round twice more: 22 x 2^-24.
bf16 grads store the norm in bf16 (8 significant bits): 2^-8 at most.
"""

import numpy as np
import pytest
import torch

from apexw_amd import _lib as L
from test_gpu_edge import _compare

pytestmark = pytest.mark.gpu

FP32_NORM = 22 * 2.0 ** -24
UNIT = {torch.bfloat16: 2.0 ** -8 + FP32_NORM, torch.float32: FP32_NORM}


def _clip_plan(params, **kw):
    from apexw_amd import ApexW
    opt = ApexW(params, lr=1e-3, weight_decay=0.1, stochastic_rounding=False, grad_centralization=True, **kw)
    opt.step()
    torch.cuda.synchronize()
    plan = next(iter(opt._plans.values()))
    assert plan.gc_fold
    return opt, plan


def _norms64(plan):
    """Each tensor's norm in float64, in parameter order, of its grad less the row means as stored."""
    out = []
    for i, p in enumerate(plan.params):
        g = p.grad
        if p.dim() >= 2:
            g = (g.reshape(p.shape[0], -1).float() - plan.gc_means[i].unsqueeze(1)).to(g.dtype)
        out.append(float(g.double().square().sum().sqrt()))
    return out


@pytest.mark.parametrize("shape", [(40, 14336), (3, 32768), (3, 32767), (3, 32769), (1, 786432), (8, 98304)])
@pytest.mark.parametrize("precision", ["compact", "8bit"])
def test_norms_of_long_rows(shape, precision):
    """Squares of one value a^2 = 1 + 0.45 x 2^-10: a single chain of n additions loses up to 0.45 x 2^-10
    of each term once its sum passes 8192."""
    print(f"long rows {precision} {shape}", flush=True)
    n = shape[0] * shape[1]
    a = (1.0 + 0.45 * 2.0 ** -10) ** 0.5
    p = torch.nn.Parameter(torch.zeros(shape, device="cuda"), requires_grad=False)
    p.grad = (torch.arange(n, device="cuda") % 2 * (2 * a) - a).float().reshape(shape)
    _, plan = _clip_plan([p], precision=precision, clip_grad_norm=1.0)
    want = _norms64(plan)[0]
    assert abs(float(plan.clip_ws[1][0]) - want) <= FP32_NORM * want


SHAPES = [(40,), (512, 1024), (4096,), (1500, 40), (33, 65), (3, 40000), (300, 2048), (64, 3, 3, 3)]


@pytest.mark.parametrize("precision", ["compact", "8bit", "ultra"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_folded_clip_norms_and_step(precision, dtype):
    """Every tensor's norm, the coefficient and the step; 8-bit tables are permuted (full-block tensors
    first), so that the row means and row lengths come from the permuted side table."""
    from oracle.clip import clip_coef
    from oracle.optim import OracleApexW
    print(f"folded clip {precision} {dtype}", flush=True)
    gen = torch.Generator().manual_seed(17)
    host = [(torch.randn(s, generator=gen) * 0.02).to(dtype) for s in SHAPES]
    # +-(1 to 1.5) about 0.5: a centralized grad near zero would make the first step's sign a rounding's
    grads = [(((1.0 + 0.5 * torch.rand(s, generator=gen)) * torch.randn(s, generator=gen).sign() + 0.5)
              * 10.0 ** (i % 3 - 3)).to(dtype) for i, s in enumerate(SHAPES)]
    gps = [torch.nn.Parameter(h.cuda(), requires_grad=False) for h in host]
    cps = [torch.nn.Parameter(h.clone(), requires_grad=False) for h in host]
    for p, q, g in zip(gps, cps, grads):
        p.grad, q.grad = g.cuda(), g.clone()
    clip = 0.25
    opt, plan = _clip_plan(gps, precision=precision, clip_grad_norm=clip)
    if precision == "8bit":
        assert plan.perm.tolist() != sorted(plan.perm.tolist())
    part, norms, coef = (t.cpu() for t in plan.clip_ws)
    want = _norms64(plan)
    for at, i in enumerate(plan.perm):
        assert abs(float(norms[at]) - want[i]) <= UNIT[dtype] * want[i], (SHAPES[i], float(norms[at]), want[i])
    total = sum(float(x) ** 2 for x in norms) ** 0.5
    assert abs(float(coef[0]) - clip / (total + 1e-6)) <= 4 * 2.0 ** -24 * float(coef[0])
    copt = OracleApexW(cps, lr=1e-3, weight_decay=0.1, stochastic_rounding=False, grad_centralization=True,
                       precision=precision, clip_grad_norm=clip)
    copt.step()
    # the oracle clips with the same coefficient (no norm fell on a rounding boundary of its dtype)
    centred = [(g.float() - g.float().reshape(g.shape[0], -1).mean(1).to(dtype).float().reshape(-1, *[1] * (g.dim() - 1)))
               .to(dtype) if g.dim() >= 2 else g for g in grads]
    assert abs(float(clip_coef(centred, clip)) - float(coef[0])) <= 1e-6 * float(coef[0])
    if dtype == torch.bfloat16:
        _compare(gps, cps, opt, copt, f"folded clip {precision}")
    else:
        for p, q in zip(gps, cps):
            # the update, near lr, takes bf16 moments in the compact precision: a unit of m (2^-8) and
            # of the root of v (2^-9)
            assert torch.allclose(p.detach().cpu(), q.detach(), rtol=1e-6, atol=2.0 ** -7 * 1e-3), tuple(p.shape)


@pytest.mark.parametrize("dtype,code", [(torch.bfloat16, L.BF16), (torch.float32, L.F32), (torch.float16, L.F16)])
@pytest.mark.parametrize("row_len", [4096, 20000, 32768, 32776])
@pytest.mark.parametrize("on_device", [False, True])
def test_row_stats_unscale_with_a_non_finite_row(dtype, code, row_len, on_device):
    """The unscale factor from the host and from a GradScaler step's device scalars; rows beyond the row
    pass's length keep what the buffer held.  The factor is a power of two, so unscaling is exact."""
    print(f"row stats unscale {dtype} {row_len} {on_device}", flush=True)
    rows, inv = 9, 2.0 ** -7
    gen = torch.Generator().manual_seed(row_len)
    g = (torch.randn(rows, row_len, generator=gen) + 0.25).to(dtype)
    g[5, row_len // 2] = float("nan")
    g[6, -1] = float("-inf")
    dg = g.cuda()
    out = torch.full((2 * rows,), -1.0, device="cuda")
    prep = np.zeros(1, dtype=L.GRAD_PREP_DTYPE)
    prep["g"], prep["out"], prep["n"], prep["row_len"], prep["dtype"] = dg.data_ptr(), out.data_ptr(), g.numel(), \
        row_len, code
    units = np.zeros(rows, dtype=L.UNIT_DTYPE)
    units["unit"] = np.arange(rows)
    up = lambda a: torch.from_numpy(a.view(np.uint8).copy()).cuda()  # noqa: E731
    dp, du = up(prep), up(units)
    amp = torch.zeros(8, device="cuda")
    amp[3] = inv                                   # apexw_amp_dyn.grad_inv_scale
    L.check(L.load().apexw_grad_row_stats(dp.data_ptr(), 1, du.data_ptr(), rows, 1.0 if on_device else inv,
                                          L.HP_SANITIZE | L.HP_UNSCALE, amp.data_ptr() if on_device else None,
                                          torch.cuda.current_stream().cuda_stream), "row stats")
    got = out.cpu()
    limit = torch.tensor(65504.0).to(dtype)
    clean = torch.where(g.isnan(), torch.zeros_like(g), torch.where(g.isinf(), limit.copysign(g), g))
    clean = (clean.float() * inv).to(dtype).double()
    mean = clean.mean(dim=1)
    ulp = {torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -23, torch.float16: 2.0 ** -11}[dtype]
    bound = mean.abs() * ulp + (row_len / 64 + 70) * 2.0 ** -24 * clean.abs().mean(dim=1)
    assert bool(((got[:rows].double() - mean).abs() <= bound).all())
    if row_len > 32768:
        assert bool((got[rows:] == -1.0).all())
        return
    want = (clean.float() - got[:rows].unsqueeze(1)).to(dtype).double().square().sum(dim=1)
    assert bool(((got[rows:].double() - want).abs() <= 40 * 2.0 ** -24 * want).all())
