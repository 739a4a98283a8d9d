"""GPU: Newton-Schulz with 128 x 128 output tiles against 256 x 256 ones, over whole steps (symmetric
products with their mirrored tiles, the addend on the matrix cores, the fused update of wide, tall and
unaligned parameters).  Every output element is the same sum in the same K order whatever tile holds it,
so parameters and results are equal bit for bit."""

import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(16, 16), (31, 40), (128, 128), (129, 200), (200, 129), (255, 257), (385, 640), (640, 385), (300, 1001)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_tiles_agree_bit_for_bit(dtype, monkeypatch):
    from apexw_amd import muon
    out = []
    for tile in (256, 128):
        monkeypatch.setattr(muon, "_tile_of", lambda *a, t=tile: t)
        gen = torch.Generator(device="cuda").manual_seed(9)
        params = [torch.nn.Parameter((torch.randn(s, device="cuda", generator=gen) * 0.02).to(dtype)) for s in SHAPES]
        grads = [(torch.randn(s, device="cuda", generator=gen) * 1e-2).to(dtype) for s in SHAPES]
        for p, g in zip(params, grads):
            p.grad = g
        opt = muon.ApexMuon(params, lr=1e-2, ns_steps=5, scale_mode="rms_matched")
        opt.keep_ns_result = True
        for _ in range(2):
            opt.step()
        ws = [w for w in opt._ws.values()]
        out.append([p.detach().clone() for p in params] + [w.rows_of(w.x[1][0]).clone() for w in ws])
    assert all(bool(torch.isfinite(x.float()).all()) for x in out[0])
    for x, y in zip(*out):
        assert torch.equal(x, y)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_kn_form_agrees_bit_for_bit(dtype, monkeypatch):
    """X as the [K x N] operand of X' = B X + a X against X^T as its [N x K] one."""
    from apexw_amd import muon
    out = []
    monkeypatch.setattr(muon, "_tile_of", lambda *a: 256)
    for most in (0, 1536):
        monkeypatch.setattr(muon, "NN_MAX_K", most)
        gen = torch.Generator(device="cuda").manual_seed(4)
        params = [torch.nn.Parameter((torch.randn(s, device="cuda", generator=gen) * 0.02).to(dtype)) for s in SHAPES]
        for p in params:
            p.grad = (torch.randn(p.shape, device="cuda", generator=gen) * 1e-2).to(dtype)
        # groups of different step counts: later iterations run on a part of the matrices
        opt = muon.ApexMuon([dict(params=params[:4], ns_steps=2), dict(params=params[4:], ns_steps=5)], lr=1e-2)
        for _ in range(2):
            opt.step()
        assert [p.nn for p in opt._ns_plans.values()] == [bool(most)]
        out.append([p.detach().clone() for p in params])
    for x, y in zip(*out):
        assert torch.equal(x, y)


def test_tile_rule():
    """Few tiles take 128, a chip's worth of long ones 256."""
    from apexw_amd.muon import NSWorkspace, _tile_of
    dev = torch.device("cuda", 0)
    small, large = [NSWorkspace(500, 500, 2, dev)], [NSWorkspace(4096, 4096, 2, dev)]
    assert [_tile_of(small, (0,), p, 256) for p in range(3)] == [128, 128, 128]
    assert [_tile_of(large, (0,), p, 256) for p in range(3)] == [256, 256, 256]
