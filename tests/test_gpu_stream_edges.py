"""Streaming kernels at the edges of their blocks and at every alignment that
decides between wide and single-element accesses."""

import pytest
import torch

from flex_shard_amd import hip_ops
from flex_shard_amd.custom_placements._copy_kernels import pack_segments_into_flat_buffer

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


@pytest.mark.parametrize("src_dtype,dst_dtype", [(torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16)])
def test_casting_copy_in(src_dtype, dst_dtype):
    """Segments of one block less, more and odd lengths, at element offsets
    0 to 5 on either side (wide accesses need multiples of four)."""
    gen = torch.Generator().manual_seed(0)
    inputs = [torch.randn(20000, generator=gen).to(src_dtype).cuda() for _ in range(2)]
    index, src, cnt, dst = [], [], [], []
    at = 0
    for which, (s, n, skip) in enumerate(
        [(0, 1024, 0), (4, 1023, 0), (8, 1025, 3), (2, 2048, 0), (1, 5, 2), (3, 3000, 1), (5, 4096, 3), (0, 1, 0), (12, 9000, 4)]
    ):
        at += skip
        index.append(which % 2), src.append(s), cnt.append(n), dst.append(at)
        at += n
    index.append(-1), src.append(0), cnt.append(1500), dst.append(at)  # zeros
    out = torch.full((at + 1600,), 7.0, dtype=dst_dtype, device="cuda")
    want = out.clone()
    for t, s, n, d in zip(index, src, cnt, dst):
        want[d : d + n] = 0 if t < 0 else inputs[t][s : s + n].to(dst_dtype)
    assert pack_segments_into_flat_buffer(inputs, index, src, cnt, dst, out) is not None
    assert torch.equal(out, want)
