"""Scaled FP8 products of few tiles: contractions shorter and longer than the
stages of operands in flight, on the tile sizes and stage counts that such
products take."""

import pytest
import torch

from flex_shard_amd import hip_ops

pytestmark = pytest.mark.gpu
E4M3 = torch.float8_e4m3fn


# 64 x 64 tiles of four stages ("deep") and of three, 128 x 128 tiles of four ("deep") and of two
@pytest.mark.parametrize(
    "m,n,tiles,with_column_scales",
    [(1, 8, "64 deep", "64 deep"), (65, 200, "64 deep", "64 deep"), (64, 16 * 1024 + 8, "64", "64 deep"),
     (1030, 2050, "64", "64"), (1090, 3080, "128 deep", "128 deep"), (1000, 5120, "128", "128")],
)
@pytest.mark.parametrize("ktiles", [1, 2, 3, 4, 5, 6, 9])
def test_every_number_of_k_tiles(device, m, n, ktiles, tiles, with_column_scales):
    """Small integers and power-of-two scales: every partial sum is exact in
    fp32 whatever the order, so the output is the one bf16 rounding of the
    exact result."""
    gen = torch.Generator().manual_seed(m + n + ktiles)
    k = 128 * ktiles
    assert hip_ops.fp8_gemm_tiles(m, n, k) == tiles
    assert hip_ops.fp8_gemm_tiles(m, n, k, column_scales=True) == with_column_scales

    def integers(rows):
        return torch.randint(-2, 3, (rows, k), generator=gen).float().to(E4M3).to(device)

    def powers(*shape):
        return torch.exp2(torch.randint(-2, 3, shape, generator=gen).float()).to(device)

    aq, bq, a_scales = integers(m), integers(n), powers(ktiles, m)
    block_scales, column_scales = powers(-(-n // 128), ktiles), powers(ktiles, n)
    blocks = [(aq[:, s : s + 128].float() @ bq[:, s : s + 128].float().T) for s in range(0, k, 128)]
    rows = [p * a_scales[kb, :, None] for kb, p in enumerate(blocks)]
    want = sum(p * block_scales[:, kb].repeat_interleave(128)[None, :n] for kb, p in enumerate(rows))
    assert torch.equal(hip_ops.fp8_gemm_1x128_128x128(aq, a_scales, bq, block_scales), want.bfloat16())
    want = sum(p * column_scales[kb][None, :] for kb, p in enumerate(rows))
    assert torch.equal(hip_ops.fp8_gemm_1x128_128x1(aq, a_scales, bq, column_scales), want.bfloat16())
