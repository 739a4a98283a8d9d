"""The step entries of general 8-bit and ultra launches: small units last, four to a group."""

import numpy as np
import pytest
import torch

from apexw_amd import _lib as L
from apexw_amd import _plan
from test_cpu_plan import _build, _opt, _params, cpu_plans  # noqa: F401 -- the fixture


def _expand(entries, n, n_fast):
    """The (tensor, unit) pairs that a launch of n entries steps, and how many entries are groups."""
    out, groups = [], 0
    for e in entries[:n]:
        if int(e["tensor"]) & L.UNIT_GROUP:
            groups += 1
            count = int(e["tensor"]) & 7
            assert 1 <= count <= 4
            first = n_fast + int(e["unit"])
            assert first >= n
            out += [tuple(map(int, x)) for x in entries[first:first + count]]
        else:
            out.append(tuple(map(int, e)))
    return out, groups


SHAPES = [(64 * 700 + 3,), (512, 1024), (50,), (40, 33), (700,), (64, 1024)]


@pytest.mark.parametrize("block_size,at_least", [(64, 0), (256, 0), (512, 0), (1024, 100), (None, 0)])
@pytest.mark.parametrize("split", [False, True])
def test_every_unit_once(cpu_plans, monkeypatch, block_size, at_least, split):  # noqa: F811
    monkeypatch.setattr(_plan, "GROUP_FROM", at_least)
    ps = _params(SHAPES, torch.bfloat16)
    opt = _opt(ps, precision="8bit", lr=1e-3, adamw_compat=True, block_size=block_size)
    plan, group = _build(opt)
    if split:
        plan.steps[::2] = 4.0
    seen = []
    monkeypatch.setattr(cpu_plans, "apexw_q8_step", lambda *a: seen.append(a) or 0, raising=False)
    tables = []
    real = _plan._upload
    monkeypatch.setattr(_plan, "_upload", lambda a, d: tables.append(real(a, d)) or tables[-1])
    plan.execute(group, seed=3)
    got, groups = [], 0
    for a in seen:
        arr = next(t for t in tables + [plan.d_step_units] if t.data_ptr() == a[2]).numpy().view(L.UNIT_DTYPE)
        pairs, k = _expand(arr, a[3], a[4] + a[5])
        got += pairs
        groups += k
        n = plan.host_table[plan.perm]["n"]
        block = plan.host_table[plan.perm]["block"].astype(np.int64)
        large = [e for e in arr[a[4] + a[5]:a[3]] if not int(e["tensor"]) & L.UNIT_GROUP]
        if k:
            assert all(min(int(n[e["tensor"]]), int(block[e["tensor"]])) > L.UNIT_GROUP_MAX for e in large)
    want = [(t, u) for t, c in enumerate(plan.unit_counts) for u in range(int(c))]
    assert sorted(got) == want
    assert groups > 0 or block_size == 1024
    assert len(seen) == (2 if split else 1)


def test_few_units_are_not_grouped(cpu_plans):  # noqa: F811
    plan, group = _build(_opt(_params([(64,)] * 300, torch.bfloat16), precision="8bit", lr=1e-3))
    plan.execute(group, seed=3)
    assert plan.d_step_units is plan.d_units and plan.n_step_units == 300
