"""The tiles of the bf16 product whose waves are laid out or whose operands are
requested in a form of their own, at ragged sizes and at contractions around the
number of k-tiles that are requested ahead.  Sums of products of small integers
are exact in fp32, so outputs are compared bit for bit."""

import ctypes

import pytest
import torch

from flex_shard_amd import _native, hip_ops

pytestmark = pytest.mark.gpu


def _integers(shape, device, gen):
    return torch.randint(-3, 4, shape, generator=gen, device=device, dtype=torch.int8).bfloat16()


def _check(device, batch, m, n, k, symmetric, tiles, offset=0):
    """alpha a b^T + beta d, with a transposed output where that is allowed, and nothing written beside them.
    ``offset``: elements by which the operands lie off a cache line."""
    assert hip_ops.gemm_tiles((batch, m, n, k, symmetric)) == (tiles,)
    gen = torch.Generator(device=device)
    gen.manual_seed(k)
    a = _integers((batch * m * k + offset,), device, gen)[offset:].view(batch, m, k)
    b = a if symmetric else _integers((batch * n * k + offset,), device, gen)[offset:].view(batch, n, k)
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


@pytest.mark.parametrize(
    "batch,m,n,k,symmetric,offset",
    [(3, 1433, 1433, k, False, offset) for k, offset in ((64, 8), (72, 0), (128, 56), (136, 0), (192, 8), (200, 0), (264, 0), (392, 0))]
    + [(2, 1968, 1968, k, True, offset) for k, offset in ((392, 0), (448, 8), (1000, 0), (1968, 0))],
)
def test_128_x_128_tiles_of_rows_that_straddle_cache_lines(device, batch, m, n, k, symmetric, offset):
    """432 and 272 tiles: some compute units have two of them, others one."""
    _check(device, batch, m, n, k, symmetric, "128", offset)


@pytest.mark.parametrize("k", [64 * 18, 64 * 19, 64 * 20, 64 * 21, 64 * 24])
@pytest.mark.parametrize("batch,m,n,symmetric,offset", [(26, 130, 257, False, 0), (26, 130, 257, False, 8), (1, 1790, 1790, True, 0)])
def test_64_x_64_tiles_of_long_contractions(device, batch, m, n, k, symmetric, offset):
    """390 and 406 tiles of 18 k-tiles and more, rows at cache lines and across them."""
    _check(device, batch, m, n, k, symmetric, "64", offset)


def test_64_x_64_tiles_of_a_contraction_that_ends_in_a_k_tile(device):
    """Rows of 1152 elements, 1144 of them summed over: whole cache lines, a last k-tile of seven chunks."""
    gen = torch.Generator(device=device)
    gen.manual_seed(5)
    a, b = _integers((26, 130, 1152), device, gen), _integers((26, 257, 1152), device, gen)
    desc, out = hip_ops._gemm_desc(a, b, None, 1.0, 0.0, None, None, False)
    desc.k = 1144
    a[:, :, 1144:], b[:, :, 1144:] = float("nan"), float("inf")  # not part of the product
    _native.check(_native.lib().fsh_gemm_bf16_nt(ctypes.byref(desc), hip_ops.stream_ptr(device)), "fsh_gemm_bf16_nt")
    want = torch.bmm(a[:, :, :1144].float(), b[:, :, :1144].float().transpose(1, 2).contiguous()).bfloat16()
    assert torch.equal(out, want)
