"""GPU: all-fp32 tensors ("full" precision) around the 512-element groups that the step takes as two runs
of 4 elements per lane: one element short of a group, whole groups, ragged tails, and a parameter that
is not 16-byte aligned (which takes the element-wise path), cold and replayed, with and without a clip.
Bars of the parity tests: 1e-6 relative plus 2^-22 of the update (at most lr)."""

import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [3, 511, 512, 513, 1023, 1024, 2047, 2048, 2049, 2560, 4100, 70001]


@pytest.mark.parametrize("clip", [None, 0.05])
@pytest.mark.parametrize("offset", [0, 1])
def test_full_precision_group_edges(clip, offset):
    from apexw_amd import ApexW
    from oracle.optim import OracleApexW
    gen = torch.Generator().manual_seed(2)
    host = [torch.randn(n, generator=gen) * 0.02 for n in SIZES]
    kw = dict(lr=1e-3, weight_decay=0.1, adamw_compat=True, precision="full", stochastic_rounding=False,
              clip_grad_norm=clip)
    gp, cp = [], []
    for h in host:
        raw = torch.zeros(h.numel() + offset, device="cuda")
        raw[offset:] = h.cuda()
        gp.append(torch.nn.Parameter(raw[offset:]))
        cp.append(torch.nn.Parameter(h.clone()))
    a, b = ApexW(gp, **kw), OracleApexW(cp, **kw)
    for _ in range(3):
        for p, q in zip(gp, cp):
            g = torch.randn(p.numel(), generator=gen) * 1e-3
            p.grad, q.grad = g.cuda(), g.clone()
        a.step()
        b.step()
    # a clip's coefficient agrees within a few fp32 units, which the quotient passes on to the update
    floor = 3 * (1e-3 * 2.0 ** -22 + (1e-3 * 2.0 ** -20 if clip else 0.0))
    for p, q in zip(gp, cp):
        x, y = p.detach().cpu(), q.detach()
        assert bool(((x - y).abs() <= 1e-6 * y.abs() + floor + 1e-9).all()), p.numel()
