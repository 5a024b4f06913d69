"""The bias of the blockwise FP8 linear inside its kernels: added in the
epilogue of the product on each tile size, its gradient summed by the pass
that quantizes the output gradient; and the one-call backward against its
parts."""

import pytest
import torch

from flex_shard_amd import hip_ops
from flex_shard_amd.blockwise_fp8.blockwise_fp8_weight import BlockwiseFp8Weight
from flex_shard_amd.blockwise_fp8.fp8_blockwise_linear import prequantized_linear

pytestmark = pytest.mark.gpu
E4M3 = torch.float8_e4m3fn


def _weight(gen, out_dim, in_dim, device):
    wq = (torch.randn(out_dim, in_dim, generator=gen) * 64).to(E4M3).to(device)
    ws = (torch.rand(-(-out_dim // 128), -(-in_dim // 128), generator=gen) * 1e-3 + 1e-4).to(device)
    return wq, ws


@pytest.mark.parametrize(
    "tokens,out_dim,in_dim,tiles",
    [
        (1, 200, 128, "64 deep"), (65, 1003, 256, "64 deep"), (1000, 2052, 512, "64"), (1091, 3081, 512, "128 deep"),
        (1001, 5123, 256, "128"), (4096, 4100, 256, "256"), (4100, 8199, 128, "256"),  # the last with half tiles
    ],
)
def test_bias_in_the_epilogue(device, tokens, out_dim, in_dim, tiles):
    """Bit for bit the separate bf16 addition, ragged rows and columns included."""
    assert hip_ops.fp8_gemm_tiles(tokens, out_dim, in_dim) == tiles
    gen = torch.Generator().manual_seed(tokens + out_dim)
    wq, ws = _weight(gen, out_dim, in_dim, device)
    xq, xs = hip_ops.act_quant_1x128(torch.randn(tokens, in_dim, generator=gen).bfloat16().to(device))
    bias = torch.randn(out_dim + 1, generator=gen).bfloat16().to(device)[1:]  # on a 2-byte boundary
    bias[0] = float("inf")
    out = torch.empty(tokens, out_dim + 3, dtype=torch.bfloat16, device=device)[:, :out_dim]
    hip_ops.fp8_gemm_1x128_128x128(xq, xs, wq, ws, out, bias=bias)
    assert torch.equal(out, hip_ops.fp8_gemm_1x128_128x128(xq, xs, wq, ws) + bias)


@pytest.mark.parametrize("tokens,out_dim,in_dim", [(1, 8, 16), (127, 130, 100), (129, 200, 136), (1000, 264, 128), (1500, 72, 384)])
def test_backward_in_one_call(device, tokens, out_dim, in_dim):
    """Every combination of wanted gradients: the products bit for bit those of
    the separate kernels, the bias gradient within the rounding of its sum."""
    gen = torch.Generator().manual_seed(tokens)
    wq, ws = _weight(gen, out_dim, in_dim, device)
    x = torch.randn(tokens, in_dim, generator=gen).bfloat16().to(device)
    g = torch.randn(tokens, out_dim, generator=gen).bfloat16().to(device)
    g8 = torch.nn.functional.pad(g, (0, -out_dim % 8))
    x8 = torch.nn.functional.pad(x, (0, -in_dim % 8))
    w16 = torch.nn.functional.pad(wq.view(torch.uint8), (0, -in_dim % 16)).view(E4M3)
    gq, gs = hip_ops.act_quant_1x128(g8)
    want_x = hip_ops.fp8_gemm_1x128_128x128_dgrad(gq, gs, hip_ops.fp8_transpose(w16), ws, in_dim=in_dim)
    want_w = hip_ops.fp8_gemm_1x128_128x1(
        *hip_ops.act_quant_128x1_transposed(g8), *hip_ops.act_quant_128x1_transposed(x8)
    )[:out_dim, :in_dim]
    exact = g.double().sum(0)
    # fp32 sums of `tokens` terms in any order, then one rounding to bf16 (8 significant bits: at most 2^-8)
    bound = tokens * 2.0**-24 * g.double().abs().sum(0) + (1 + 2.0**-8) * 2.0**-8 * exact.abs() + 2.0**-100
    for needs in [(1, 1, 1), (1, 1, 0), (1, 0, 1), (0, 1, 1), (0, 1, 0), (1, 0, 0), (0, 0, 1)]:
        weight = BlockwiseFp8Weight(wq, ws, 128, orig_dtype=torch.bfloat16, requires_grad=bool(needs[1]))
        bias = torch.zeros(out_dim, dtype=torch.bfloat16, device=device).requires_grad_(bool(needs[2]))
        x_in = x.clone().requires_grad_(bool(needs[0]))
        out = prequantized_linear(x_in, weight, bias)
        out.backward(g)
        assert (x_in.grad is not None, weight.grad is not None, bias.grad is not None) == tuple(map(bool, needs))
        if needs[0]:
            assert torch.equal(x_in.grad, want_x)
        if needs[1]:
            assert torch.equal(weight.grad, want_w)
        if needs[2]:
            assert bias.grad.shape == bias.shape and ((bias.grad.double() - exact).abs() <= bound).all()


def test_no_graph_and_graph_give_the_same_output(device):
    """Without gradients the product takes the activation in one form only; a
    bias of another type or a broadcast one is added outside the kernel."""
    gen = torch.Generator().manual_seed(3)
    wq, ws = _weight(gen, 256, 256, device)
    weight = BlockwiseFp8Weight(wq, ws, 128, orig_dtype=torch.bfloat16, requires_grad=True)
    x = torch.randn(4, 30, 256, generator=gen).bfloat16().to(device)
    wide = torch.randn(512, generator=gen)
    for bias in (None, wide[:256].bfloat16().to(device), wide.bfloat16().to(device)[::2], wide[:256].to(device), wide[:1].bfloat16().to(device)):
        tracked = prequantized_linear(x, weight, bias)
        with torch.no_grad():
            plain = prequantized_linear(x, weight, bias)
        assert tracked.grad_fn is not None and plain.grad_fn is None
        base = prequantized_linear(x, weight, None).detach()
        want = base if bias is None else base + bias
        assert plain.dtype == want.dtype and torch.equal(plain, want) and torch.equal(tracked.detach(), want)
