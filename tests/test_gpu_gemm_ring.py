"""The operand ring of the 256 x 256 tiles: contractions of fewer k-tiles than
the ring holds, and of every position its slots can end in, in both operand
forms, on resident and on separate workgroups."""

import pytest
import torch

from flex_shard_amd import hip_ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,side", [(2, 4096), (13, 1024)])  # 512 tiles: more than the compute units; 208: fewer
@pytest.mark.parametrize("ktiles", [1, 2, 3, 4, 5, 6, 7, 8, 11])
def test_every_ring_position_in_both_operand_forms(device, batch, side, ktiles):
    """Sums of products of small integers are exact in fp32, so the outputs are the one bf16 rounding."""
    assert hip_ops.gemm_tiles((batch, side, side, 64 * ktiles)) == ("256",)
    gen = torch.Generator(device=device)
    gen.manual_seed(ktiles)
    a, b = (torch.randint(-3, 4, (batch, 64 * ktiles, side), generator=gen, device=device).bfloat16() for _ in range(2))
    ref = torch.bmm(a.float().transpose(1, 2).contiguous(), b.float()).bfloat16()
    assert torch.equal(hip_ops.gemm_nt(a, b, k_major=True), ref)
    assert torch.equal(hip_ops.gemm_nt(a.transpose(1, 2).contiguous(), b.transpose(1, 2).contiguous()), ref)
