"""The bias gradient of the FP8 linear is linear in the output gradient, and a
backward of the backward goes through it, also where the weight gradient is
wanted and the quantizer's pass could have summed the gradient."""

import pytest
import torch

from flex_shard_amd.blockwise_fp8 import BlockwiseFp8Weight, Fp8BlockwiseGemms, prequantized_linear


def test_sum_is_torchs_under_a_graph(monkeypatch):
    from flex_shard_amd import hip_ops

    asked = []

    def backward(grad, wq, ws, in_dim, x_runs, needs_x_grad, needs_weight_grad, needs_bias_grad):
        asked.append(needs_bias_grad)
        tokens, out = grad.shape
        bias = torch.full((out,), 7.0, dtype=grad.dtype) if needs_bias_grad else None
        return torch.zeros(tokens, in_dim, dtype=grad.dtype), torch.zeros(out, in_dim, dtype=grad.dtype), bias

    monkeypatch.setattr(hip_ops, "fp8_linear_backward", backward)
    weight = BlockwiseFp8Weight(torch.zeros(24, 16).to(torch.float8_e4m3fn), torch.ones(1, 1), 128)
    runs = (torch.zeros(16, 128).to(torch.float8_e4m3fn), torch.ones(1, 16))
    for requires_grad, grad_mode in ((False, True), (True, False), (True, True)):
        grad = torch.arange(48.0).view(2, 24).bfloat16().requires_grad_(requires_grad)
        with torch.set_grad_enabled(grad_mode):
            _, _, bias = Fp8BlockwiseGemms(128)._backward(grad, None, weight, True, True, True, runs)
        assert bias.requires_grad == (requires_grad and grad_mode)
        assert torch.equal(bias.detach(), grad.detach().sum(0) if bias.requires_grad else torch.full_like(bias, 7.0))
    assert asked == [True, True, False]


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [1, 64, 130])
def test_second_backward_through_the_bias_gradient(device, tokens):
    gen = torch.Generator().manual_seed(tokens)
    weight = BlockwiseFp8Weight(
        torch.randn(200, 136, generator=gen).to(torch.float8_e4m3fn).to(device), torch.ones(2, 2, device=device), 128,
        requires_grad=True,
    )
    x = torch.randn(tokens, 136, generator=gen).bfloat16().to(device).requires_grad_()
    bias = torch.randn(200, generator=gen).bfloat16().to(device).requires_grad_()
    out = prequantized_linear(x, weight, bias)
    grad_out = torch.randn(tokens, 200, generator=gen).bfloat16().to(device).requires_grad_()
    _, _, grad_bias = torch.autograd.grad(out, [x, weight, bias], grad_out, create_graph=True)
    factor = torch.randn(200, generator=gen).bfloat16().to(device)
    (second,) = torch.autograd.grad(grad_bias, grad_out, factor)
    assert torch.equal(second, factor.expand(tokens, 200))
