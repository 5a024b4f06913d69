"""Forward-mode derivatives of the FP8 linear are not implemented, and a call
that would need one is refused with gradients on or off: without them the
layer's function is skipped, which must not drop a tangent silently."""

import pytest
import torch
from torch.autograd import forward_ad

from flex_shard_amd.blockwise_fp8 import BlockwiseFp8Weight, prequantized_linear


class _HostGemms:
    def forward(self, x, weight):
        return x @ weight.fp8_data.float().t()


def _weight():
    return BlockwiseFp8Weight(torch.ones(8, 16).to(torch.float8_e4m3fn), torch.ones(1, 1), 128, orig_dtype=torch.float32)


@pytest.mark.parametrize("dual", ["x", "bias"])
@pytest.mark.parametrize("grad_mode", [True, False])
def test_a_dual_tensor_is_refused(grad_mode, dual):
    x, bias = torch.randn(4, 16), torch.randn(8)
    with torch.set_grad_enabled(grad_mode), forward_ad.dual_level():
        if dual == "x":
            x = forward_ad.make_dual(x, torch.ones_like(x))
        else:
            bias = forward_ad.make_dual(bias, torch.ones_like(bias))
        with pytest.raises(NotImplementedError):
            prequantized_linear(x, _weight(), bias, _HostGemms())


@pytest.mark.parametrize("grad_mode", [True, False])
def test_plain_tensors_in_a_dual_level_are_multiplied(grad_mode):
    x = torch.randn(4, 16)
    with torch.set_grad_enabled(grad_mode), forward_ad.dual_level():
        out = prequantized_linear(x, _weight(), None, _HostGemms())
        assert forward_ad.unpack_dual(out).tangent is None
    assert torch.equal(out, x @ torch.ones(16, 8))
