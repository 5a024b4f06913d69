"""Newton-Schulz on the 256 x 256 tiles where sizes are not whole tiles: edge
tiles of a few rows and columns, contractions that end in every octet of a
k-tile (bit for bit against the small tiles), tall, wide and square, products
that take the large tiles on their own, and the update behind them."""

import pytest
import torch

from flex_shard_amd import hip_ops
from flex_shard_amd.dist_muon import OwnedMuon
from flex_shard_amd.dist_muon.muon_math import _apply_muon_update, _prepare_muon_input
from flex_shard_amd.testing import seeded_normal

pytestmark = pytest.mark.gpu
COEFFS = (3.4445, -4.7750, 2.0315)


@pytest.mark.parametrize("shape", [(24, 1000, 1000), (60, 504, 1000), (12, 1528, 1288), (30, 1032, 768), (8, 2056, 2056), (24, 1016, 2040)])
@pytest.mark.parametrize("steps", [1, 2])
def test_ragged_sizes_against_64_bits(device, shape, steps):
    assert hip_ops.newton_schulz_large_tiles(shape, steps=steps) == (True,)
    batch, rows, cols = shape
    guard = 4096
    x = torch.full((batch * rows * cols + 2 * guard,), 7.0, dtype=torch.bfloat16, device=device)
    mine = x[guard:-guard].view(shape)
    mine.copy_(seeded_normal(shape, 1.0, rows + cols, device))
    start = mine.double()
    nbytes = hip_ops.newton_schulz_workspace_bytes(*shape)
    workspace = torch.full((nbytes + 4096,), 0x55, dtype=torch.uint8, device=device)
    hip_ops.newton_schulz_multi([(mine, workspace[:nbytes])], COEFFS, steps, 1e-7)
    assert (x[:guard] == 7).all() and (x[-guard:] == 7).all() and (workspace[nbytes:] == 0x55).all()
    _check(mine, start, steps, (0, batch - 1))


# Short sides that end in octet 0 .. 7 of a k-tile; long ones in 1, 4, 7, 2, 5, 0, 3, 6.
OCTETS = [(26, 704, 712), (26, 672, 648), (26, 656, 696), (26, 720, 664), (26, 672, 680), (26, 704, 680), (26, 688, 728), (26, 752, 696)]
PRODUCTS = [(product, last) for product in (0, 1, 2) for last in (False, True)]


def _tiles(shape):
    return {hip_ops.newton_schulz_product_tiles(shape, product=product, last=last)[0] for product, last in PRODUCTS}


@pytest.mark.parametrize("shape", OCTETS)
def test_every_octet_equals_the_small_tiles_bit_for_bit(device, shape):
    """The batch fills the large tiles; one of its matrices alone takes small ones."""
    assert _tiles(shape) == {"256"} and "256" not in _tiles((1, *shape[1:]))
    together = seeded_normal(shape, 1.0, sum(shape), device)
    alone = {b: together[b : b + 1].clone() for b in (0, 11, 25)}
    hip_ops.newton_schulz_multi([(together, None)], COEFFS, 3, 1e-7)
    for b, x in alone.items():
        hip_ops.newton_schulz_multi([(x, None)], COEFFS, 3, 1e-7)
        assert torch.equal(together[b], x[0]), b


# Short sides that end in octet 2, 4, 6, 7 (wide) and 1, 3, 5, 2 (tall).
FREE = [(2, 1936, 2200), (2, 2016, 2200), (2, 2096, 2200), (2, 1976, 2200), (2, 2216, 2056), (2, 2216, 2008), (2, 2216, 1960), (2, 2216, 1936)]


@pytest.mark.parametrize("shape", FREE)
def test_third_product_alone_on_large_tiles(device, shape):
    """Few matrices iterate on the small tiles; their third product, with its
    transposed output, may still take the large ones.  One matrix of the two
    declines that, with the same bits."""
    assert hip_ops.newton_schulz_large_tiles(shape) == (False,)
    tiles = {q: hip_ops.newton_schulz_product_tiles(shape, product=q[0], last=q[1])[0] for q in PRODUCTS}
    assert {q for q, kind in tiles.items() if kind == "256"} == {(2, False), (2, True)}
    assert "256" not in _tiles((1, *shape[1:]))
    together = seeded_normal(shape, 1.0, sum(shape), device)
    alone = together[1:].clone()
    start = together.double()
    hip_ops.newton_schulz_multi([(together, None)], COEFFS, 3, 1e-7)
    hip_ops.newton_schulz_multi([(alone, None)], COEFFS, 3, 1e-7)
    assert torch.equal(together[1], alone[0])
    _check(together, start, 3, (0,))


def _check(mine, start, steps, which):
    rows, cols = mine.shape[1:]
    for b in which:
        ref = start[b] if rows <= cols else start[b].T.contiguous()
        ref = ref / ref.norm()
        for _ in range(steps):
            g = ref @ ref.T
            ref = COEFFS[0] * ref + (COEFFS[1] * g + COEFFS[2] * g @ g) @ ref
        ref = ref if rows <= cols else ref.T
        diff = mine[b].double() - ref
        # five roundings to bf16 a step, each 2^-9 of values that the polynomial's slope (3.4 at most) amplifies
        assert diff.norm() <= 2e-2 * ref.norm()
        assert diff.abs().max() <= 0.1 * ref.abs().max()  # no element of an edge stands out


def test_update_behind_ragged_large_tiles(device):
    """Shapes that are multiples of 8 take the update in the last product's epilogue, padded ones the separate kernel."""
    shapes = [(1000, 1000)] * 24 + [(999, 1001)] * 24
    assert hip_ops.newton_schulz_large_tiles((24, 1000, 1000), (24, 1000, 1008)) == (True, True)
    mine = [seeded_normal(s, 0.02, i, device) for i, s in enumerate(shapes)]
    theirs = [p.clone() for p in mine]
    grads = [seeded_normal(s, 1.0, 100 + i, device) for i, s in enumerate(shapes)]
    OwnedMuon(mine, lr=2e-3, weight_decay=0.05).step(grads)
    momenta = [torch.zeros_like(p) for p in theirs]
    batches = [torch.zeros(24, 1000, cols, dtype=torch.bfloat16, device=device) for cols in (1000, 1008)]
    for i, (rows, cols) in enumerate(shapes):
        u = torch.empty(rows, cols, dtype=torch.bfloat16, device=device)
        _prepare_muon_input(grads[i], momenta[i], momentum=0.95, nesterov=True, out=u)
        batches[i // 24][i % 24, :rows, :cols] = u
    hip_ops.newton_schulz_multi([(b, None) for b in batches], COEFFS, 5, 1e-7)
    for i, (rows, cols) in enumerate(shapes):
        d = batches[i // 24][i % 24, :rows, :cols].contiguous()
        _apply_muon_update(theirs[i], d, lr=2e-3, weight_decay=0.05, adjust_lr_fn=None, compute_matrix_shape=(rows, cols))
        assert torch.equal(mine[i], theirs[i]), i
