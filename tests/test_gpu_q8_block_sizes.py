"""GPU: INT8 and ultra blocks at the edges of the general 8-bit kernel's split (a workgroup per block, 8
elements per thread): every block size, tensors one element around them, one wave, four waves and
ragged tails, zero grads and a tiny eps (which takes the IEEE sequences), against the CPU oracle with
stochastic rounding off.  Bars as in the parity tests: 1 code, 1 bf16 unit, 1e-6 relative for scales
and fp32."""

import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [(64,), (65,), (127,), (255,), (511,), (513,), (1023,), (1025,), (2047,), (2048,), (2049,), (4095,), (6145,),
         (16, 3, 3, 3), (33, 67), (5, 1639)]


@pytest.mark.parametrize("precision", ["8bit", "ultra"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("eps", [1e-8, 1e-16])
def test_block_edges_match_oracle(precision, dtype, eps):
    from apexw_amd import ApexW
    from oracle.optim import OracleApexW
    gen = torch.Generator().manual_seed(5)
    # fewer than 8 tensors per optimizer, which keeps fp32 8-bit parameters fp32
    for at in range(0, len(SIZES), 6):
        shapes = SIZES[at:at + 6]
        host = [(torch.randn(s, generator=gen) * 0.02).to(dtype) for s in shapes]
        grads = [(torch.randn(s, generator=gen) * 1e-3).to(dtype) for s in shapes]
        grads[0].zero_()
        kw = dict(lr=1e-3, weight_decay=0.1, eps=eps, adamw_compat=True, precision=precision,
                  stochastic_rounding=False)
        gp = [torch.nn.Parameter(h.cuda(), requires_grad=False) for h in host]
        cp = [torch.nn.Parameter(h.clone(), requires_grad=False) for h in host]
        for p, q, g in zip(gp, cp, grads):
            p.grad, q.grad = g.cuda(), g.clone()
        a, b = ApexW(gp, **kw), OracleApexW(cp, **kw)
        a.step()
        b.step()
        for p, q in zip(gp, cp):
            x, y = p.detach().cpu().float(), q.detach().float()
            # the update, near lr, is rounded to the parameter's dtype before it is subtracted
            unit = 2.0 ** -7 if dtype == torch.bfloat16 else 1e-6
            assert bool(((x - y).abs() <= unit * y.abs() + unit * 2e-3).all()), (precision, tuple(p.shape))
            for k, v in a.state[p].items():
                if not (torch.is_tensor(v) and v.is_cuda):
                    continue
                w = b.state[q][k]
                if v.dtype in (torch.int8, torch.uint8) and k in ("exp_avg", "exp_avg_sq"):
                    d = (v.cpu().to(torch.int32) - w.to(torch.int32)).abs()
                    assert int(d.max()) <= 1, (k, tuple(p.shape))
                else:
                    rel = 2.0 ** -8 if v.dtype == torch.bfloat16 else 1e-6
                    assert torch.allclose(v.cpu().float().reshape(-1), w.float().reshape(-1), rtol=rel, atol=1e-30), k
