"""Edges of the memory-bound kernels around the optimizer's products: the
normalization's division over the exponents, fp32 masters of few and of odd
elements."""

import pytest
import torch

from flex_shard_amd import hip_ops
from flex_shard_amd.dist_muon import OwnedMuon, _apply_muon_update, _prepare_muon_input

pytestmark = pytest.mark.gpu
COEFFS = (3.4445, -4.7750, 2.0315)


def _normalized(x):
    """bf16(x / max(bf16(norm), eps)) and the norm, whose fp32 sum is too far
    from a bf16 rounding boundary for its order to matter."""
    exact = x.float().square().sum().sqrt() if not x.double().square().sum() < 1e38 else x.double().square().sum().sqrt()
    norm = max(exact.float().bfloat16().item(), torch.tensor(1e-7).bfloat16().item()) if exact == exact else float("nan")
    return (x.float() / torch.tensor(norm, device=x.device)).bfloat16()


@pytest.mark.parametrize("shape", [(8, 8), (72, 200), (200, 72), (1000, 1544)])
@pytest.mark.parametrize("case", ["usual", "tiny", "mixed", "huge", "overflow", "zero", "inf", "nan"])
def test_normalization_divides(device, shape, case):
    """Bit for bit the fp32 division rounded to bf16."""
    gen = torch.Generator().manual_seed(shape[0])
    x = torch.randn(shape, generator=gen)
    if case == "mixed":  # exponents down to the subnormals beside ordinary values
        x = x * torch.exp2(-torch.randint(0, 132, shape, generator=gen).float())
    x = x * {"tiny": 2.0**-110, "huge": 2.0**52, "overflow": 2.0**100, "zero": 0.0}.get(case, 1.0)
    x = x.bfloat16()
    if case == "inf":
        x[-1, -1] = float("inf")
    if case == "nan":
        x[0, 0] = float("nan")
    x = x.to(device)
    want = _normalized(x)
    got = hip_ops.newton_schulz(x.clone(), COEFFS, 0, 1e-7)
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got[~got.isnan()], want[~got.isnan()])


@pytest.mark.parametrize("case", ["usual", "tiny", "huge", "zero"])
@pytest.mark.parametrize("shape", [(8, 8), (72, 200), (200, 72)])
def test_normalization_keeps_the_sign_of_zero(device, shape, case):
    """The int16 views are equal, zeros of either sign among the values."""
    gen = torch.Generator().manual_seed(shape[1])
    x = torch.randn(shape, generator=gen) * {"tiny": 2.0**-110, "huge": 2.0**52, "zero": 0.0}.get(case, 1.0)
    x = x.bfloat16()
    zero = torch.rand(shape, generator=gen) < 0.25
    x[zero] = torch.where(torch.rand(shape, generator=gen) < 0.5, 0.0, -0.0).bfloat16()[zero]
    x = x.to(device)
    want = _normalized(x)
    assert want[want == 0].signbit().any() and not want[want == 0].signbit().all()
    got = hip_ops.newton_schulz(x.clone(), COEFFS, 0, 1e-7)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


# whole slices, slices that end inside a wave, less than one wave, odd rows and columns
@pytest.mark.parametrize("shapes", [[(8, 8), (8, 520), (64, 1000)], [(1024, 1544), (1032, 72)], [(130, 77), (512, 512)]])
def test_fp32_masters_equal_the_per_matrix_kernels(device, shapes):
    gen = torch.Generator().manual_seed(3)
    start = [torch.randn(s, generator=gen).to(device) * 0.02 for s in shapes]
    mine, theirs = [p.clone() for p in start], [p.clone() for p in start]
    momenta = [torch.zeros_like(p) for p in theirs]
    opt = OwnedMuon(mine, lr=2e-3, weight_decay=0.05)
    for step in range(2):
        grads = [torch.randn(s, generator=gen).to(device) for s in shapes]
        opt.step(grads)
        for i, s in enumerate(shapes):
            batch = torch.empty((1, *s), dtype=torch.bfloat16, device=device)
            _prepare_muon_input(grads[i], momenta[i], momentum=0.95, nesterov=True, out=batch[0])
            hip_ops.newton_schulz(batch, COEFFS, 5, 1e-7)
            _apply_muon_update(theirs[i], batch[0], lr=2e-3, weight_decay=0.05, adjust_lr_fn=None, compute_matrix_shape=s)
            assert torch.equal(opt.momentum_buffers[i], momenta[i]), f"momentum {s} at step {step}"
            assert torch.equal(mine[i], theirs[i]), f"parameter {s} at step {step}"
