"""The tiles of the bf16 product whose waves are laid out or whose operands are
requested in a form of their own, at ragged sizes and at contractions around the
number of k-tiles that are requested ahead.  Sums of products of small integers
are exact in fp32, so outputs are compared bit for bit."""

import pytest
import torch

from flex_shard_amd import hip_ops

pytestmark = pytest.mark.gpu


def _integers(shape, device, gen):
    return torch.randint(-3, 4, shape, generator=gen, device=device, dtype=torch.int8).bfloat16()


def _check(device, batch, m, n, k, symmetric, tiles):
    """alpha a b^T + beta d, with a transposed output where that is allowed, and nothing written beside them."""
    assert hip_ops.gemm_tiles((batch, m, n, k, symmetric)) == (tiles,)
    gen = torch.Generator(device=device)
    gen.manual_seed(k)
    a = _integers((batch, m, k), device, gen)
    b = a if symmetric else _integers((batch, n, k), device, gen)
    d = _integers((batch, m, n), device, gen)
    if symmetric:
        d = d + d.transpose(1, 2)
    pad = 256
    bufs = [torch.full((batch * m * n + 2 * pad,), 7.0, dtype=torch.bfloat16, device=device) for _ in range(2)]
    c, ct = bufs[0][pad:-pad].view(batch, m, n), bufs[1][pad:-pad].view(batch, n, m)
    hip_ops.gemm_nt(a, b, d=d.contiguous(), alpha=0.5, beta=2.0, out=c, out_t=None if symmetric else ct, symmetric=symmetric)
    want = (0.5 * torch.bmm(a.float(), b.float().transpose(1, 2).contiguous()) + 2.0 * d.float()).bfloat16()
    assert torch.equal(c, want)
    assert torch.equal(ct, want.transpose(1, 2).contiguous()) if not symmetric else (ct == 7).all()
    assert all((buf[:pad] == 7).all() and (buf[-pad:] == 7).all() for buf in bufs)


@pytest.mark.parametrize(
    "batch,m,n,k,symmetric",
    [(3, 1433, 1433, 1000, False), (3, 1159, 2000, 1000, False), (20, 200, 1500, 1000, False), (7, 1283, 1283, 1544, True),
     (1, 3000, 3000, 3000, True), (1, 2400, 2400, 2432, False)],
)
def test_256_x_128_tiles(device, batch, m, n, k, symmetric):
    _check(device, batch, m, n, k, symmetric, "256x128")
