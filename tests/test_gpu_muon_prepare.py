"""GPU: the grouped Muon preparation (momentum, then normalised work matrices of several matrices in two
launches) at the edges of its chunks, 64 x 64 tiles, 8-element vectors and 32 x 32 panels, in both
layouts and for unaligned grads, against the same torch ops.

Bars: the momentum is one FMA on an exactly representable product's rounding (bit-equal); the work
matrix is bf16(bf16(s) / d), where d may differ by one bf16 unit when the fp32 norms' summation order
rounds it the other way, so an element differs by at most two bf16 units (2^-7 relative)."""

import numpy as np
import pytest
import torch

from apexw_amd import _lib as L
from apexw_amd.muon import _from_panels

pytestmark = pytest.mark.gpu

SHAPES = [(16, 16), (31, 33), (64, 64), (65, 130), (130, 65), (257, 40), (17, 2049), (700, 768), (1000, 530)]


@pytest.mark.parametrize("layout", [L.LAYOUT_ROWS, L.LAYOUT_PANEL])
@pytest.mark.parametrize("gdt,code", [(torch.float32, L.F32), (torch.bfloat16, L.BF16), (torch.float16, L.F16)])
@pytest.mark.parametrize("nesterov", [0, 1])
@pytest.mark.parametrize("offset", [0, 1])
def test_grouped_prepare_matches_torch(layout, gdt, code, nesterov, offset):
    lib = L.load()
    gen = torch.Generator(device="cuda").manual_seed(7)
    mu, eps = 0.95, 1e-7
    items, keep, units = [], [], ([], [])
    for k, (r, c) in enumerate(SHAPES):
        buf = torch.randn(r, c, device="cuda", generator=gen)
        raw = torch.randn(r * c + offset, device="cuda", generator=gen).to(gdt)
        raw[offset] = float("nan")
        g = raw[offset:].view(r, c)
        m, n = min(r, c), max(r, c)
        ldx, ldxt = -(-n // 256) * 256, -(-m // 256) * 256
        x = torch.zeros(ldxt, ldx, dtype=torch.bfloat16, device="cuda")
        xt = torch.zeros(ldx, ldxt, dtype=torch.bfloat16, device="cuda")
        part = torch.empty(int(lib.apexw_muon_workspace_floats(r, c)), device="cuda")
        keep.append((buf, buf.clone(), g, x, xt, part))
        items.append((buf.data_ptr(), g.data_ptr(), x.data_ptr(), xt.data_ptr(), part.data_ptr(), r, c, ldx, ldxt, mu,
                      1.0 - mu, code, layout, nesterov, 0))
        for which in (0, 1):
            units[which].extend((k, u) for u in range(int(lib.apexw_muon_prepare_units(r, c, which))))
    table = np.array(items, dtype=L.MUON_ITEM_DTYPE)
    assert lib.apexw_check_muon_items(table.ctypes.data, len(table)) == 0
    up = lambda a: torch.from_numpy(a.view(np.uint8).copy()).cuda()  # noqa: E731
    dt, du = up(table), [up(np.array(u, dtype=L.UNIT_DTYPE)) for u in units]
    L.check(lib.apexw_muon_prepare_grouped(dt.data_ptr(), len(table), du[0].data_ptr(), len(units[0]), du[1].data_ptr(),
                                           len(units[1]), eps, 1.0, None, torch.cuda.current_stream().cuda_stream),
            "prepare")
    torch.cuda.synchronize()
    for (r, c), (buf, old, g, x, xt, _) in zip(SHAPES, keep):
        gf = torch.nan_to_num(g.float(), nan=0.0, posinf=65504.0, neginf=-65504.0)
        ref = (old * np.float32(mu)).add(gf, alpha=float(np.float32(1.0 - mu)))
        assert torch.equal(buf, ref)
        s = (torch.lerp(gf, ref, mu) if nesterov else ref).bfloat16()
        d = (s.double().norm().bfloat16() + eps).bfloat16()
        want = (s.float() / d.float()).bfloat16()
        wide = want if r <= c else want.t()
        for out, w in ((x, wide), (xt, wide.t())):
            got = (_from_panels(out) if layout == L.LAYOUT_PANEL else out).float()
            w = w.float()
            assert bool(((got[:w.shape[0], :w.shape[1]] - w).abs() <= 2.0 ** -7 * w.abs()).all())
            got[:w.shape[0], :w.shape[1]] = 0.0
            assert not bool(got.any()), "padding written"
