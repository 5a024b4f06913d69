"""An owner with more shape groups than one native call takes steps in several
calls; a step that any of them can't take updates nothing."""

import pytest
import torch

from flex_shard_amd import hip_ops
from flex_shard_amd.dist_muon import OwnedMuon, muon_math


class _Plan:
    """Records steps; refuses what has a negative first element."""

    MAX_GROUPS = 2
    stepped: list = []

    def __init__(self, groups, device):
        self.batches = self.workspaces = [None] * len(groups)

    def check(self, params, momenta, grads):
        if any(g.flatten()[0] < 0 for group in grads for g in group):
            raise ValueError("refused")

    def step(self, params, momenta, grads, **kwargs):
        self.check(params, momenta, grads)
        _Plan.stepped.append([tuple(g.shape) for group in grads for g in group])


@pytest.mark.parametrize("bad", range(5))
def test_all_plans_are_asked_before_the_first_steps(monkeypatch, bad):
    monkeypatch.setattr(hip_ops, "MuonStepPlan", _Plan)
    monkeypatch.setattr(muon_math, "_require_master_gpu", lambda *tensors: None)
    monkeypatch.setattr(_Plan, "stepped", [])
    opt = OwnedMuon([torch.zeros(8, n + 1) for n in range(5)])
    grads = [torch.ones_like(p) for p in opt.params]
    grads[bad].neg_()
    with pytest.raises(ValueError, match="refused"):
        opt.step(grads)
    assert _Plan.stepped == []
    grads[bad].neg_()
    opt.step(grads)
    assert _Plan.stepped == [[(8, 1), (8, 2)], [(8, 3), (8, 4)], [(8, 5)]]


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [0, 16, 17])
def test_misaligned_gradient_of_any_group(device, bad):
    gen = torch.Generator().manual_seed(bad)
    shapes = [(8 * (i + 1), 24) for i in range(18)]
    assert len(shapes) > hip_ops.MuonStepPlan.MAX_GROUPS
    start = [(torch.randn(s, generator=gen) * 0.02).bfloat16().to(device) for s in shapes]
    grads = [torch.randn(s, generator=gen).bfloat16().to(device) for s in shapes]
    params = [p.clone() for p in start]
    opt = OwnedMuon(params)
    shifted = list(grads)
    rows, cols = shapes[bad]
    storage = torch.zeros(rows * cols + 8, dtype=torch.bfloat16, device=device)
    shifted[bad] = storage[1 : 1 + rows * cols].view(rows, cols)
    with pytest.raises(ValueError, match="aligned"):
        opt.step(shifted)
    assert all(torch.equal(a, b) for a, b in zip(params, start))
    assert not any(m.any() for m in opt.momentum_buffers)
    opt.step(grads)
    for i, (p, g) in enumerate(zip(start, grads)):
        alone = OwnedMuon([p])
        alone.step([g])
        assert torch.equal(params[i], p) and torch.equal(opt.momentum_buffers[i], alone.momentum_buffers[0])
