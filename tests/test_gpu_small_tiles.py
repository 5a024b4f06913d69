"""The small tiles of the bf16 product where their pipeline can go wrong:
contractions of fewer, as many and one more k-tiles than are requested ahead,
whole and ending inside a k-tile, and rows so far apart that a tile's offsets
need 64 bits.  Sums of products of small integers are exact in fp32, so outputs are
compared bit for bit."""

import ctypes

import pytest
import torch

from flex_shard_amd import _native, hip_ops

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
def test_contractions_on_both_sides_of_the_choice_of_wide_offsets(device, k):
    """Through the public entry: rows that long are contiguous there, and few of them fit a test."""
    gen = torch.Generator(device=device)
    gen.manual_seed(1)
    a, b = _integers((9, k), device, gen, 1), _integers((5, k), device, gen, 1)  # sums below 2^24
    want = a.double() @ b.double().t().contiguous()
    assert torch.equal(hip_ops.gemm_nt(a, b), want.to(torch.float32).bfloat16())


class _Strided:
    """Integers in the first k columns of rows that lie ld elements apart in one large allocation."""

    def __init__(self, device, gen, rows, k, ld):
        self.storage = torch.empty((rows - 1) * ld + k, dtype=torch.bfloat16, device=device)
        self.ld, self.values = ld, _integers((rows, k), device, gen, 3)
        self.storage.as_strided((rows, k), (ld, 1)).copy_(self.values)


def _describe(a, b, batch=1):
    """A descriptor of a b^T whose operands are :class:`_Strided`, or tensors; all matrices of a batch are the same."""
    at, bt = (t.values if isinstance(t, _Strided) else t for t in (a, b))
    desc, out = hip_ops._gemm_desc(at.expand(batch, *at.shape).contiguous(), bt.expand(batch, *bt.shape).contiguous(), None, 1.0,
                                   0.0, None, None, False)
    desc.a_dev, desc.b_dev = (t.storage.data_ptr() if isinstance(t, _Strided) else t.data_ptr() for t in (a, b))
    desc.lda, desc.ldb = (t.ld if isinstance(t, _Strided) else t.shape[1] for t in (a, b))
    desc.stride_a = desc.stride_b = 0
    return desc, out, (at.float() @ bt.float().t().contiguous()).bfloat16()


# Offsets of 32 bits would take row r + 64 of a tile for row r.
ALIASED = 1 << 25


@pytest.mark.parametrize("rows,k,both", [(130, 72, False), (130, 136, True), (120, 64, True), (65, 200, False)])
def test_offsets_of_a_tile_beyond_4_gib(device, rows, k, both):
    gen = torch.Generator(device=device)
    gen.manual_seed(k)
    wide, narrow = _Strided(device, gen, rows, k, ALIASED), _integers((70, k), device, gen, 3)
    for a, b in ((wide, wide),) if both else ((wide, narrow), (narrow, wide)):
        desc, out, want = _describe(a, b)
        _native.check(_native.lib().fsh_gemm_bf16_nt(ctypes.byref(desc), hip_ops.stream_ptr(device)), "fsh_gemm_bf16_nt")
        assert torch.equal(out[0], want)


def test_offsets_of_a_tile_just_below_2_gib(device):
    """256 x 128 tiles: row 255 lies 2^31 - 2^23 - 4080 bytes behind row 0."""
    assert hip_ops.gemm_tiles((3, 1433, 1433, 1000)) == ("256x128",)
    gen = torch.Generator(device=device)
    gen.manual_seed(2)
    a, b = _Strided(device, gen, 1433, 1000, (1 << 22) - 8), _integers((1433, 1000), device, gen, 3)
    desc, out, want = _describe(a, b, batch=3)
    _native.check(_native.lib().fsh_gemm_bf16_nt(ctypes.byref(desc), hip_ops.stream_ptr(device)), "fsh_gemm_bf16_nt")
    assert all(torch.equal(c, want) for c in out)


@pytest.mark.parametrize("at", [0, 1, 2])
def test_one_problem_of_a_launch_has_wide_rows(device, at):
    gen = torch.Generator(device=device)
    gen.manual_seed(at)
    problems = []
    for i, (m, n, k) in enumerate(((130, 257, 200), (100, 70, 136), (200, 129, 72))):
        a = _Strided(device, gen, m, k, ALIASED) if i == at else _integers((m, k), device, gen, 3)
        problems.append((a, _integers((n, k), device, gen, 3)))
    described = [_describe(a, b) for a, b in problems]
    descs = (_native.GemmDesc * 3)(*(desc for desc, _, _ in described))
    _native.check(_native.lib().fsh_gemm_bf16_nt_group(descs, 3, hip_ops.stream_ptr(device)), "fsh_gemm_bf16_nt_group")
    for _, out, want in described:
        assert torch.equal(out[0], want)
