"""The FP8 tiles over contractions that use every slot of a k-tile's chunks, the
last k-tiles at every place.  256 x 256: three of the early ones by two of the
late ones, six k-tiles; 16 of the 272 tiles are cut into halves, whose chunks
are all early.  Smaller ones: as many slots as k-tiles in flight (two to four)
and one more of the early ones, twenty k-tiles at the most."""

import pytest
import torch

from flex_shard_amd import hip_ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ktiles", [2, 3, 6, 7, 8, 9, 10, 11, 13])
@pytest.mark.parametrize("column_scales", [False, True])
def test_every_place_of_a_k_tile(device, ktiles, column_scales):
    _check(device, 4090, 4120, ktiles, column_scales, "256")


@pytest.mark.parametrize("column_scales", [False, True])
@pytest.mark.parametrize(
    "m,n,tiles,ktiles",
    [(m, n, tiles, ktiles) for m, n, tiles in ((130, 1000, "64 deep"), (1090, 3080, "128 deep")) for ktiles in (7, 12, 19, 20, 21, 22, 23, 24)]
    + [(m, n, tiles, ktiles) for m, n, tiles in ((1030, 2050, "64"), (1923, 2180, "128")) for ktiles in (7, 8, 10, 11, 12)],
)
def test_every_place_of_a_k_tile_in_small_tiles(device, m, n, tiles, ktiles, column_scales):
    _check(device, m, n, ktiles, column_scales, tiles)


def _check(device, m, n, ktiles, column_scales, tiles):
    """Small integers and powers of two: exact in fp32, one rounding to bf16."""
    k = 128 * ktiles
    assert hip_ops.fp8_gemm_tiles(m, n, k, column_scales=column_scales) == tiles
    gen = torch.Generator(device=device)
    gen.manual_seed(ktiles)
    a, b = (torch.randint(-3, 4, (rows, k), generator=gen, device=device).float() for rows in (m, n))
    powers = lambda *shape: torch.randint(-2, 3, shape, generator=gen, device=device).float().exp2()  # noqa: E731
    a_scales = powers(ktiles, m)
    b_scales = powers(ktiles, n) if column_scales else powers(-(-n // 128), ktiles)
    per_row = b_scales.T if column_scales else b_scales.repeat_interleave(128, 0)[:n]
    left = (a.view(m, -1, 128) * a_scales.T.unsqueeze(-1)).view(m, k)
    right = (b.view(n, -1, 128) * per_row.unsqueeze(-1)).view(n, k)
    product = hip_ops.fp8_gemm_1x128_128x1 if column_scales else hip_ops.fp8_gemm_1x128_128x128
    got = product(a.to(torch.float8_e4m3fn), a_scales, b.to(torch.float8_e4m3fn), b_scales)
    assert torch.equal(got, (left.double() @ right.double().T).bfloat16())
