"""The launch rules of the products as their host-only queries report them."""

import pytest

from flex_shard_amd import hip_ops


def test_every_kind_of_tile_is_chosen_somewhere():
    bf16 = {
        hip_ops.gemm_tiles((batch, m, m, k, symmetric))[0]
        for batch in (1, 7, 24) for m in (40, 520, 1283, 2048, 3000) for k in (64, 520, 1544) for symmetric in (False, True)
    }
    assert bf16 == {"64", "128", "128 deep", "256x128", "256"}
    fp8 = {
        hip_ops.fp8_gemm_tiles(m, n, k, column_scales=scales)
        for m in (1, 1000, 1090, 8192) for n in (200, 2052, 3080, 5120, 14336) for k in (128, 4096, 33152) for scales in (False, True)
    }
    assert fp8 == set(hip_ops.GEMM_TILES) - {"256x128"}


def test_problems_of_one_call_share_the_choice():
    """Whole 256 x 256 tiles go together or not at all, ragged problems beside
    them; more problems than a launch holds are looked at launch by launch."""
    ragged, few, many = (2, 264, 136, 72), (8, 1280, 1280, 64), (40, 1536, 1536, 192)
    assert hip_ops.gemm_tiles(ragged, many, few) == ("64", "256", "256")
    assert len(set(hip_ops.gemm_tiles(few, ragged))) == 1 and hip_ops.gemm_tiles() == ()
    assert hip_ops.gemm_tiles(*[(1, 64, 64, 64)] * 8, (1, 1920, 1928, 264)) == ("64",) * 8 + ("128 deep",)
    assert hip_ops.newton_schulz_large_tiles((24, 7168, 2048), (24, 2048, 2048), (1, 64, 96)) == (True, True, False)
    assert hip_ops.newton_schulz_large_tiles((1, 2048, 2048)) == (False,)
    assert hip_ops.newton_schulz_large_tiles((24, 7168, 2048), steps=0) == (False,)


@pytest.mark.parametrize(
    "long,short,tiles",
    [((13, 384, 384, 3560, True), (1, 2432, 2432, 2432, True), "128 deep"), ((4, 1024, 1024, 4096, True), (8, 1024, 1024, 1024, True), "128 deep"),
     ((8, 768, 768, 3072, True), (10, 768, 768, 768, True), "128"), ((2, 1280, 1280, 1280, True), (8, 832, 832, 832, True), "128")],
)
def test_short_tiles_beside_long_ones_count_by_their_length(long, short, tiles):
    """More than 256 tiles of 128 x 128, by length up to 0.86 of a round of the long ones and more."""
    assert hip_ops.gemm_tiles(long, short) == (tiles, tiles)


def test_third_product_takes_large_tiles_within_one_round_only():
    """Problems that iterate on the small tiles: their third product joins the
    256 x 256 ones up to a round of 256 of them, and only where that is faster."""
    third = lambda *shapes, **kw: hip_ops.newton_schulz_product_tiles(*shapes, product=2, **kw)  # noqa: E731
    assert hip_ops.newton_schulz_large_tiles((2, 2048, 3072)) == hip_ops.newton_schulz_large_tiles((3, 2048, 3072)) == (False,)
    assert third((2, 2048, 3072)) == third((2, 3072, 2048)) == third((1, 3072, 3072), last=True) == ("256",)  # 192 and 144 tiles
    assert third((3, 2048, 3072)) == third((3, 3072, 2048)) == ("256x128",)  # 288 tiles
    assert third((1, 2248, 2248)) == third((1, 2600, 2200)) == ("256x128",)  # 81 and 99: too few to gain by it
    assert third((24, 2048, 2048), (1, 64, 96)) == ("256", "64") and third() == ()
    for product in (0, 1):
        assert hip_ops.newton_schulz_product_tiles((2, 2048, 3072), product=product) != ("256",)


def test_bad_sizes_are_refused():
    for shape, kw in (((1, 64, 64), {"product": 3}), ((1, 64, 64), {"product": 0, "steps": 0}), ((1, 64, 60), {"product": 0}), ((0, 64, 64), {"product": 0})):
        with pytest.raises(RuntimeError, match="newton_schulz"):
            hip_ops.newton_schulz_product_tiles(shape, **kw)
    for sizes in ((0, 8, 8, 8), (1, 8, 8, 12)):
        with pytest.raises(RuntimeError, match="gemm"):
            hip_ops.gemm_tiles(sizes)
    with pytest.raises(RuntimeError, match="symmetric"):
        hip_ops.gemm_tiles((1, 8, 16, 8, True))
    with pytest.raises(RuntimeError, match="bad list"):
        hip_ops.gemm_tiles(*[(1, 8, 8, 8)] * 17)
    for sizes in ((0, 8, 128), (8, 8, 100)):
        with pytest.raises(RuntimeError, match="bad sizes"):
            hip_ops.fp8_gemm_tiles(*sizes)
