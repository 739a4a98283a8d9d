"""GPU: small units stepped in groups, a wave each, equal a workgroup each bit for bit (stochastic rounding
too: the noise is keyed by tensor and element), and the per-parameter update likewise."""

import pytest
import torch

pytestmark = pytest.mark.gpu

# few and many blocks, ragged tails, larger blocks and full-block tensors among them, tensors under 64 elements
SHAPES = [(64 * 300 + 7,), (512, 1024), (37,), (40, 33), (700,), (5000,), (12,), (3, 64, 65)]


def _run(monkeypatch, grouped, precision, dtype, sr, trainable=False, **kw):
    from apexw_amd import ApexW, _plan
    monkeypatch.setattr(_plan, "GROUP_FROM", 0 if grouped else 1 << 40)
    gen = torch.Generator().manual_seed(3)
    torch.manual_seed(5)                       # the optimizer draws its rounding seed from torch's generator
    ps = [torch.nn.Parameter((torch.randn(s, generator=gen) * 0.02).to(dtype).cuda(), requires_grad=trainable)
          for s in SHAPES]
    opt = ApexW(ps, lr=1e-3, weight_decay=0.1, precision=precision, stochastic_rounding=sr, **kw)
    for _ in range(3):
        grads = [(torch.randn(s, generator=gen) * 1e-3).to(dtype).cuda() for s in SHAPES]
        if trainable:                          # stepped inside the backward
            sum((p * g).sum() for p, g in zip(ps, grads)).backward()
        else:
            for p, g in zip(ps, grads):
                p.grad = g
        opt.step()
    torch.cuda.synchronize()
    return ps, opt


@pytest.mark.parametrize("precision,kw", [("8bit", dict(block_size=64)), ("8bit", dict(block_size=256)),
                                          ("8bit", dict(block_size=512, grad_centralization=True, clip_grad_norm=0.1)),
                                          ("8bit", {}), ("8bit", dict(cautious=True)), ("ultra", {})])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("sr", [False, True])
def test_grouped_units_equal_single_ones(monkeypatch, precision, kw, dtype, sr):
    print(f"unit groups {precision} {kw} {dtype} {sr}", flush=True)
    one, a = _run(monkeypatch, False, precision, dtype, sr, **kw)
    many, b = _run(monkeypatch, True, precision, dtype, sr, **kw)
    plan = next(iter(b._plans.values()))
    assert plan.n_step_units < plan.n_units      # some share an entry
    for p, q in zip(one, many):
        assert torch.equal(p, q), tuple(p.shape)
        for k, v in a.state[p].items():
            if torch.is_tensor(v):
                assert torch.equal(v, b.state[q][k]), (tuple(p.shape), k)


def test_grouped_units_inside_the_backward(monkeypatch):
    """The automatic in-backward 8-bit batches take the same entries."""
    print("unit groups in backward", flush=True)
    one, a = _run(monkeypatch, False, "8bit", torch.bfloat16, True, trainable=True, block_size=64)
    many, b = _run(monkeypatch, True, "8bit", torch.bfloat16, True, trainable=True, block_size=64)
    for p, q in zip(one, many):
        assert torch.equal(p, q), tuple(p.shape)
