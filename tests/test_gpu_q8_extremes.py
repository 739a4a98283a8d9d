"""GPU: quantized steps at the ends of the fp32 range, against the CPU oracle with stochastic rounding off."""

import pytest
import torch

pytestmark = pytest.mark.gpu

FLT_MAX = torch.finfo(torch.float32).max
SCALE = FLT_MAX / 127.0 * (1.0 - 2.0 ** -20)      # 127 SCALE is finite, 128 SCALE is not


def _pair(shape, grad, dtype=torch.float32, **kw):
    """The same one-tensor optimizer on the GPU and in the oracle, parameters at zero."""
    from apexw_amd import ApexW
    from oracle.optim import OracleApexW
    kw = dict(lr=1e-3, weight_decay=0.0, adamw_compat=True, stochastic_rounding=False, **kw)
    # 8-bit: plain shards whose grads the program assigns (trainable ones step inside the backward)
    gp = torch.nn.Parameter(torch.zeros(shape, dtype=dtype, device="cuda"), requires_grad=False)
    cp = torch.nn.Parameter(torch.zeros(shape, dtype=dtype), requires_grad=False)
    gp.grad, cp.grad = grad.to(dtype).cuda(), grad.to(dtype).clone()
    return gp, cp, ApexW([gp], **kw), OracleApexW([cp], **kw)


@pytest.mark.parametrize("precision,factored,shape", [("8bit", False, (4096,)), ("8bit", False, (4097,)),
                                                      ("ultra", False, (64, 64)), ("ultra", False, (63, 65)),
                                                      ("8bit", True, (256, 2048)), ("8bit", True, (256, 1536))])
def test_int8_moments_at_the_top_of_the_range(precision, factored, shape):
    """INT8 codes whose scale times 128 overflows while code times scale does not: the moments decode to
    finite values.  The next m and p are single fp32 operations per element: 1e-6 relative."""
    print(f"int8 top of range {precision} {factored} {shape}", flush=True)
    gen = torch.Generator().manual_seed(7)
    gp, cp, a, b = _pair(shape, torch.zeros(shape), precision=precision, factored_v=factored)
    a.step()
    b.step()
    sa, sb = a.state[gp], b.state[cp]
    assert bool(sa.get("is_factored_v", False)) == factored
    codes = torch.randint(-127, 128, (sb["exp_avg"].numel(),), generator=gen, dtype=torch.int32).to(torch.int8)
    codes[::64] = 127
    for st in (sa, sb):
        st["exp_avg"].copy_(codes.view(st["exp_avg"].shape).view(st["exp_avg"].dtype))
        st["exp_avg_scales"].fill_(SCALE)
        if factored:
            st["exp_avg_sq_row"].fill_(1e34)
            st["exp_avg_sq_col"].fill_(1e34)
        elif precision == "ultra":
            st["exp_avg_sq"].fill_(1e37)
        else:
            st["exp_avg_sq"].fill_(255)
            st["exp_avg_sq_scales"].fill_(1e37)
    a.step()
    b.step()
    x, y = gp.detach().cpu(), cp.detach()
    assert bool(torch.isfinite(y).all()) and float(y.abs().max()) > 0.0
    assert torch.allclose(x, y, rtol=2e-6, atol=0.0)
    assert torch.allclose(sa["exp_avg_scales"].cpu().reshape(-1), sb["exp_avg_scales"].reshape(-1), rtol=1e-6, atol=0.0)
    d = sa["exp_avg"].cpu().reshape(-1).to(torch.int32) - sb["exp_avg"].reshape(-1).to(torch.int32)
    assert int(d.abs().max()) <= 1


@pytest.mark.parametrize("precision,shape", [("8bit", (4096,)), ("8bit", (4099,)), ("ultra", (64, 64)),
                                             ("ultra", (63, 65))])
def test_subnormal_second_moments(precision, shape):
    """Grads of 1e-17 to 1e-20 leave second moments below the smallest normal number beside normal ones
    and zeros, under a denominator eps of one unit of 2^-63: fp32 parameters equal the oracle's IEEE root
    and quotient bit for bit."""
    print(f"subnormal v {precision} {shape}", flush=True)
    gen = torch.Generator().manual_seed(11)
    mag = 10.0 ** (-17.0 - 3.0 * torch.rand(shape, generator=gen, dtype=torch.float64))
    grad = (mag * torch.randn(shape, generator=gen, dtype=torch.float64).sign()).float()
    grad.view(-1)[::7] = 0.0
    # the step's eps is eps sqrt(1 - beta2) = 1.26e-12
    gp, cp, a, b = _pair(shape, grad, precision=precision, eps=4e-11)
    a.step()
    b.step()
    x, y = gp.detach().cpu(), cp.detach()
    assert int((y != 0).sum()) > y.numel() // 2
    assert torch.equal(x, y), int((x != y).sum())
