"""Gradient accumulation on both sides of the size from which the accumulator streams."""

import pytest
import torch

from flex_shard_amd import hip_ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("numel", [(5 << 24) - 1, 5 << 24, (5 << 24) + 1027])
def test_two_microbatches_around_the_streaming_size(device, numel):
    gen = torch.Generator(device=device)
    gen.manual_seed(numel)
    guard = 64
    buf = torch.full((numel + 2 * guard,), 7.0, device=device)
    acc = buf[guard:-guard]
    first, second = (torch.randn(numel, generator=gen, device=device).bfloat16() for _ in range(2))
    hip_ops.accumulate_grad(acc, first, overwrite=True)
    assert torch.equal(acc, first.float())
    hip_ops.accumulate_grad(acc, second)
    assert torch.equal(acc, first.float() + second.float())
    assert (buf[:guard] == 7).all() and (buf[-guard:] == 7).all()
