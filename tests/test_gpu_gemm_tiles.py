"""The tile kernels of the bf16 NT product at the sizes where they can go
wrong: ragged rows and columns, contractions that end inside a k-tile or hold
fewer k-tiles than the pipeline is deep, every tile size the launch rule
chooses between (the rule is asked which one a case takes), and several
problems in one launch."""

import pytest
import torch

from flex_shard_amd import hip_ops

pytestmark = pytest.mark.gpu

CASES = [
    # 64 x 64 tiles
    (1, 1, 1, 8), (1, 64, 64, 64), (1, 65, 63, 72), (2, 130, 257, 136), (1, 129, 127, 520), (3, 33, 300, 248),
    # 128 x 128 tiles, operands requested four k-tiles ahead (240 tiles)
    (1, 1920, 1928, 264), (1, 1923, 1837, 392), (1, 1920, 1920, 576),
    # 64 x 64 tiles, more than the chip holds at once (2304 and 2304 tiles)
    (32, 520, 500, 456), (32, 513, 511, 520),
    # 128 x 128 tiles, two workgroups per compute unit
    (32, 512, 512, 512), (9, 1544, 1288, 72),
    # 256 x 256 tiles, resident workgroups
    (20, 1024, 1280, 1024),
]


def _operands(batch, m, n, k, device, seed):
    gen = torch.Generator(device=device)
    gen.manual_seed(seed)
    a = torch.randn(batch, m, k, generator=gen, device=device).bfloat16()
    b = torch.randn(batch, n, k, generator=gen, device=device).bfloat16()
    d = torch.randn(batch, m, n, generator=gen, device=device).bfloat16()
    return a, b, d


def _close(got, ref):
    # one rounding to bf16 (half an ulp, 2^-9 of the value) of an fp32 sum whose own error, k 2^-24 of the
    # sum of magnitudes (about k for these operands), stays below 2e-2 up to k = 1024
    return torch.allclose(got.double(), ref, rtol=2.0**-8, atol=2e-2)


@pytest.mark.parametrize("batch,m,n,k", CASES)
def test_ragged_products_with_addend_and_transposed_output(device, batch, m, n, k):
    a, b, d = _operands(batch, m, n, k, device, m + n + k)
    pad = 512
    bufs = [torch.full((batch * m * n + 2 * pad,), 7.0, dtype=torch.bfloat16, device=device) for _ in range(2)]
    c, ct = bufs[0][pad:-pad].view(batch, m, n), bufs[1][pad:-pad].view(batch, n, m)
    hip_ops.gemm_nt(a, b, d=d, alpha=0.5, beta=2.0, out=c, out_t=ct)
    ref = 0.5 * torch.bmm(a.double(), b.double().transpose(1, 2).contiguous()) + 2.0 * d.double()
    assert _close(c, ref)
    assert torch.equal(ct, c.transpose(1, 2).contiguous())
    for buf in bufs:
        assert (buf[:pad] == 7).all() and (buf[-pad:] == 7).all()


@pytest.mark.parametrize("batch,n,k", [(1, 70, 40), (4, 300, 200), (40, 648, 328), (1, 1928, 136)])
def test_ragged_symmetric_products_with_a_diagonal_term(device, batch, n, k):
    a, _, _ = _operands(batch, n, n, k, device, n + k)
    got = hip_ops.gemm_nt(a, a, symmetric=True, diag_add=1.5)
    assert torch.equal(got, got.transpose(1, 2).contiguous())
    ref = torch.bmm(a.double(), a.double().transpose(1, 2).contiguous()) + 1.5 * torch.eye(n, device=device, dtype=torch.float64)
    assert _close(got, ref)
    assert torch.equal(got, hip_ops.gemm_nt(a, a, diag_add=1.5))  # the same sums, every tile computed


@pytest.mark.parametrize(
    "tiles,batch,m,n,k",
    [
        ("64", 2, 130, 257, 136), ("64", 32, 513, 511, 520), ("128", 32, 512, 512, 512), ("128", 8, 337, 1500, 200),
        ("128 deep", 1, 1923, 1837, 392), ("256x128", 3, 1433, 1433, 1000), ("256x128", 3, 1159, 2000, 1000),
        ("256x128", 20, 200, 1500, 1000), ("256", 7, 1536, 1280, 64), ("256", 20, 1024, 1280, 1024),
    ],
)
def test_small_integers_on_every_kind_of_tile(device, tiles, batch, m, n, k):
    """Sums of products of small integers are exact in fp32 whatever the order,
    so the outputs are the one bf16 rounding of the exact result."""
    assert hip_ops.gemm_tiles((batch, m, n, k)) == (tiles,)
    a, b, d = (t.round().clamp(-3, 3) for t in _operands(batch, m, n, k, device, m + n + k))
    pad = 512
    bufs = [torch.full((batch * m * n + 2 * pad,), 7.0, dtype=torch.bfloat16, device=device) for _ in range(2)]
    c, ct = bufs[0][pad:-pad].view(batch, m, n), bufs[1][pad:-pad].view(batch, n, m)
    hip_ops.gemm_nt(a, b, d=d, alpha=0.5, beta=2.0, out=c, out_t=ct)
    want = (0.5 * torch.bmm(a.float(), b.float().transpose(1, 2).contiguous()) + 2.0 * d.float()).bfloat16()
    assert torch.equal(c, want)
    assert torch.equal(ct, want.transpose(1, 2).contiguous())
    for buf in bufs:
        assert (buf[:pad] == 7).all() and (buf[-pad:] == 7).all()


@pytest.mark.parametrize(
    "tiles,batch,n,k",
    [("64", 4, 300, 200), ("128", 6, 1536, 192), ("256x128", 7, 1283, 1544), ("256x128", 1, 3000, 3000), ("256", 10, 1536, 128)],
)
def test_small_integers_in_symmetric_products(device, tiles, batch, n, k):
    assert hip_ops.gemm_tiles((batch, n, n, k, True)) == (tiles,)
    a, _, d = (t.round().clamp(-3, 3) for t in _operands(batch, n, n, k, device, n + k))
    d = torch.triu(d) + torch.triu(d, 1).transpose(1, 2)
    pad = 512
    buf = torch.full((batch * n * n + 2 * pad,), 7.0, dtype=torch.bfloat16, device=device)
    c = buf[pad:-pad].view(batch, n, n)
    hip_ops.gemm_nt(a, a, d=d, alpha=0.5, beta=2.0, symmetric=True, diag_add=1.5, out=c)
    want = 0.5 * torch.bmm(a.float(), a.float().transpose(1, 2).contiguous()) + 2.0 * d.float()
    assert torch.equal(c, (want + 1.5 * torch.eye(n, device=device)).bfloat16())
    assert (buf[:pad] == 7).all() and (buf[-pad:] == 7).all()


def test_more_problems_than_one_launch_holds(device):
    problems = []
    for i in range(11):
        a, b, _ = _operands(1 + i % 3, 40 + 37 * i, 250 - 19 * i, 8 * (1 + 3 * i), device, i)
        problems.append({"a": a, "b": b})
    for q, out in zip(problems, hip_ops.gemm_nt_group(problems)):
        assert torch.equal(out, hip_ops.gemm_nt(q["a"], q["b"]))
        assert _close(out, torch.bmm(q["a"].double(), q["b"].double().transpose(1, 2).contiguous()))


@pytest.mark.parametrize("master", [torch.bfloat16, torch.float32])
def test_muon_step_on_odd_shapes_equals_the_per_matrix_kernels(device, master):
    """Matrices whose rows are not whole 16-byte vectors, beside ones whose
    are, in the batched step: more shape groups than one call takes, one
    matrix larger than a block's slice, odd addresses."""
    from flex_shard_amd.dist_muon import OwnedMuon
    from flex_shard_amd.dist_muon.muon_math import _apply_muon_update, _compute_muon_direction, _prepare_muon_input

    gen = torch.Generator(device=device)
    gen.manual_seed(5)
    shapes = [(1, 1), (7, 9), (64, 72), (130, 257), (257, 130), (33, 8), (8, 33)] + [(20 + i, 40) for i in range(12)]

    def odd_view(shape):  # starts one element into its storage where the shape allows it
        off = 0 if shape[0] % 8 == 0 and shape[1] % 8 == 0 else 1
        return torch.randn(shape[0] * shape[1] + off, generator=gen, device=device).to(master)[off:].view(shape)

    params, grads = [odd_view(s) for s in shapes], [odd_view(s) for s in shapes]
    want, momenta = [p.clone() for p in params], [torch.zeros_like(p) for p in params]
    opt = OwnedMuon(params, lr=0.02)
    for _ in range(2):
        opt.step(grads)
        for p, m, g in zip(want, momenta, grads):
            d = _prepare_muon_input(g, m, momentum=0.95, nesterov=True, out=torch.empty(p.shape, dtype=torch.bfloat16, device=device))
            _compute_muon_direction(d)
            _apply_muon_update(p, d, lr=0.02, weight_decay=0.1, adjust_lr_fn=None, compute_matrix_shape=p.shape)
    for shape, p, w, m, n in zip(shapes, params, want, opt.momentum_buffers, momenta):
        assert torch.equal(p, w), shape
        assert torch.equal(m, n), shape
