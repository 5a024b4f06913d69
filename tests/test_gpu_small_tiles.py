"""The small tiles of the bf16 product where their pipeline can go wrong:
contractions of fewer, as many and one more k-tiles than are requested ahead,
whole and ending inside a k-tile, and rows so long that a tile's offsets need
64 bits.  Sums of products of small integers are exact in fp32, so outputs are
compared bit for bit."""

import pytest
import torch

from flex_shard_amd import hip_ops

pytestmark = pytest.mark.gpu


def _integers(shape, device, gen, high):
    return torch.randint(-high, high + 1, shape, generator=gen, device=device, dtype=torch.int8).bfloat16()


@pytest.mark.parametrize("k", [64, 72, 128, 192, 200, 256, 264, 320, 328, 392])
@pytest.mark.parametrize("batch,m,n", [(2, 130, 257), (26, 130, 257), (25, 130, 257), (9, 1546, 1288), (1, 1923, 1837), (3, 1433, 1433)])
def test_pipeline_depths(device, batch, m, n, k):
    tiles = hip_ops.gemm_tiles((batch, m, n, k))
    assert tiles == ({2: "64", 25: "64", 26: "64", 9: "128", 1: "128 deep", 3: "128"}[batch],)
    gen = torch.Generator(device=device)
    gen.manual_seed(k)
    a, b, d = (_integers((batch, *s), device, gen, 3) for s in ((m, k), (n, k), (m, n)))
    pad = 256
    bufs = [torch.full((batch * m * n + 2 * pad,), 7.0, dtype=torch.bfloat16, device=device) for _ in range(2)]
    c, ct = bufs[0][pad:-pad].view(batch, m, n), bufs[1][pad:-pad].view(batch, n, m)
    hip_ops.gemm_nt(a, b, d=d, alpha=0.5, beta=2.0, out=c, out_t=ct)
    want = (0.5 * torch.bmm(a.float(), b.float().transpose(1, 2).contiguous()) + 2.0 * d.float()).bfloat16()
    assert torch.equal(c, want)
    assert torch.equal(ct, want.transpose(1, 2).contiguous())
    assert all((buf[:pad] == 7).all() and (buf[-pad:] == 7).all() for buf in bufs)


@pytest.mark.parametrize("k", [(1 << 22) - 8, 1 << 22, (1 << 22) + 72])
def test_rows_on_both_sides_of_32_bit_offsets(device, k):
    gen = torch.Generator(device=device)
    gen.manual_seed(1)
    a, b = _integers((9, k), device, gen, 1), _integers((5, k), device, gen, 1)  # sums below 2^24
    want = a.double() @ b.double().t().contiguous()
    assert torch.equal(hip_ops.gemm_nt(a, b), want.to(torch.float32).bfloat16())
