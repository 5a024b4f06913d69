"""Newton-Schulz on the 256 x 256 tiles where sizes are not whole tiles: edge
tiles of a few rows and columns, contractions that end in any octet of a
k-tile, tall, wide and square, and the update behind them."""

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


@pytest.mark.parametrize("shape", [(1, 2248, 2248), (1, 3072, 3072), (1, 2600, 2200)])
def test_third_product_alone_on_large_tiles(device, shape):
    """Few matrices iterate on the small tiles; their third product, with its
    transposed output, may still take the large ones."""
    assert hip_ops.newton_schulz_large_tiles(shape) == (False,)
    mine = seeded_normal(shape, 1.0, sum(shape), device)
    start = mine.double()
    hip_ops.newton_schulz_multi([(mine, None)], COEFFS, 3, 1e-7)
    _check(mine, start, 3, (0,))


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
