"""Streaming kernels at the edges of their blocks and at every alignment that
decides between wide and single-element accesses."""

import pytest
import torch

from flex_shard_amd import hip_ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("acc_offset,grad_offset", [(0, 0), (0, 4), (4, 8), (1, 0), (0, 2), (3, 3)])
@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 4096, 5000])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_accumulate(n, acc_offset, grad_offset, dtype):
    gen = torch.Generator().manual_seed(n)
    first, second = ((torch.randn(n + 16, generator=gen)).to(dtype).cuda()[grad_offset : grad_offset + n] for _ in range(2))
    base = torch.full((n + 16,), 7.0, device="cuda")
    acc = base[acc_offset : acc_offset + n]
    hip_ops.accumulate_grad(acc, first, overwrite=True)
    assert torch.equal(acc, first.float())
    hip_ops.accumulate_grad(acc, second)
    assert torch.equal(acc, first.float() + second.float())
    assert (base[:acc_offset] == 7).all() and (base[acc_offset + n :] == 7).all()
