"""Tiles whose rows are not 16-byte friendly: the quantizer's unaligned path
beside aligned chunks of the same launch, against the oracle."""

import pytest
import torch

from flex_shard_amd import hip_ops
from oracle import cport

pytestmark = pytest.mark.gpu

SHAPES = [(257, 343), (128, 256), (3, 1), (130, 129), (1, 7), (300, 136), (129, 8), (64, 250), (2, 513)]


@pytest.mark.parametrize("count", [1, 3, 9])  # of up to eight and of more chunks
@pytest.mark.parametrize("gap", [0, 1, 6])  # bytes between the chunks' data: their payload positions
@pytest.mark.parametrize("master", [torch.bfloat16, torch.float32])
def test_unaligned_chunks_beside_aligned_ones(device, count, gap, master):
    gen = torch.Generator().manual_seed(count + gap)
    weights = [(torch.randn(s, generator=gen) * 0.02).to(master) for s in SHAPES[:count]]
    weights[-1][-1, -1] = 3.0e38  # the largest element is a row's last
    at, specs, spans = 5, [], []
    for w in weights:
        spans.append((at, w.numel()))
        at += w.numel() + gap
    scales_at = (at + 3) // 4 * 4
    for w, (start, _) in zip(weights, spans):
        kind = hip_ops.SRC_BF16 if master == torch.bfloat16 else hip_ops.SRC_F32_AS_BF16
        specs.append(hip_ops.QuantChunkSpec(w.to(device), start, scales_at, kind))
        scales_at += 4 * -(-w.shape[0] // 128) * -(-w.shape[1] // 128)
    payload = torch.full((scales_at + 9,), 0xAA, dtype=torch.uint8, device=device)
    hip_ops.quantize_pack(specs, payload, ((0, 2), (scales_at + 1, scales_at + 6)), 128)
    want = torch.full((scales_at + 9,), 0xAA, dtype=torch.uint8)
    want[0:2] = 0
    want[scales_at + 1 : scales_at + 6] = 0
    for w, spec in zip(weights, specs):
        q, s = cport.quantize_blockwise(w.bfloat16(), 128)
        want[spec.qdata_offset :][: w.numel()] = q.reshape(-1)
        want[spec.scale_offset :][: 4 * s.numel()] = s.contiguous().reshape(-1).view(torch.uint8)
    assert torch.equal(payload.cpu(), want)


@pytest.mark.parametrize("master", [torch.bfloat16, torch.float32])
def test_nan_poisons_its_tile_alone(device, master):
    w = torch.ones(130, 129).to(master)
    w[3, 4] = float("nan")
    payload = torch.zeros(130 * 129 + 2 + 16, dtype=torch.uint8, device=device)
    kind = hip_ops.SRC_BF16 if master == torch.bfloat16 else hip_ops.SRC_F32_AS_BF16
    hip_ops.quantize_pack([hip_ops.QuantChunkSpec(w.to(device), 0, 130 * 129 + 2, kind)], payload, ((0, 0), (0, 0)), 128)
    q, s = payload[: 130 * 129].view(130, 129).cpu(), payload[130 * 129 + 2 :].cpu().view(torch.float32)
    assert ((q[:128, :128] & 0x7F) == 0x7F).all() and (q[:, 128] == 0x7E).all() and (q[128:] == 0x7E).all()
    assert s[0].isnan() and (s[1:] == 1 / 448).all()
