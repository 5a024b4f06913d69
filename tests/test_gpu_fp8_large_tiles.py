"""The 256 x 256 FP8 tiles with contractions of one k-tile and a few, ragged
edges and a last round of half tiles, both scale forms."""

import pytest
import torch

from flex_shard_amd import hip_ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n", [(6000, 4120), (4096, 4120)])  # 408 tiles; 272, whose last 16 are cut into halves
@pytest.mark.parametrize("k", [128, 256, 384, 640])
@pytest.mark.parametrize("column_scales", [False, True])
def test_small_integers_with_powers_of_two_as_scales(device, m, n, k, column_scales):
    """Every sum is exact in fp32, so the outputs are the one bf16 rounding."""
    assert hip_ops.fp8_gemm_tiles(m, n, k, column_scales=column_scales) == "256"
    gen = torch.Generator(device=device)
    gen.manual_seed(k)
    a, b = (torch.randint(-3, 4, (rows, k), generator=gen, device=device).float() for rows in (m, n))
    exponents = lambda *shape: torch.randint(-2, 3, shape, generator=gen, device=device).float().exp2()  # noqa: E731
    a_scales = exponents(k // 128, m)
    aq, bq = a.to(torch.float8_e4m3fn), b.to(torch.float8_e4m3fn)
    left = (a.view(m, -1, 128) * a_scales.T.unsqueeze(-1)).view(m, k)
    if column_scales:
        b_scales = exponents(k // 128, n)
        right = (b.view(n, -1, 128) * b_scales.T.unsqueeze(-1)).view(n, k)
        got = hip_ops.fp8_gemm_1x128_128x1(aq, a_scales, bq, b_scales)
    else:
        b_scales = exponents(-(-n // 128), k // 128)
        right = (b.view(n, -1, 128) * b_scales.repeat_interleave(128, 0)[:n].unsqueeze(-1)).view(n, k)
        got = hip_ops.fp8_gemm_1x128_128x128(aq, a_scales, bq, b_scales)
    assert torch.equal(got, (left.double() @ right.double().T).bfloat16())
