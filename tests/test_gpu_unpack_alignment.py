"""The 128-block unpack at widths and byte offsets that are not multiples of
eight: whole groups of eight go out unaligned, a row's last bytes one by one."""

import pytest
import torch

from flex_shard_amd import hip_ops

pytestmark = pytest.mark.gpu
E4M3 = torch.float8_e4m3fn


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,in_dim", [(1, 7), (129, 8), (130, 9), (16, 127), (257, 136), (100, 1001)])
def test_unpack_of_any_width_and_offset(device, rows, in_dim, dtype):
    """Two chunks; compact bytes exact, values the fp32 product rounded once,
    bytes around the destinations untouched."""
    gen = torch.Generator().manual_seed(rows * in_dim)
    data = torch.randint(0, 256, (2, rows, in_dim), dtype=torch.uint8, generator=gen)
    data[(data & 0x7F) == 0x7F] = 0x3C
    tiles = (-(-rows // 128), -(-in_dim // 128))
    scales = torch.rand(2, *tiles, generator=gen) * 1e-2 + 1e-4
    n, ns = rows * in_dim, tiles[0] * tiles[1]
    want = torch.stack([
        data[c].view(E4M3).float() * scales[c].repeat_interleave(128, 0)[:rows].repeat_interleave(128, 1)[:, :in_dim] for c in range(2)
    ]).to(dtype)
    for lead in (0, 1, 4, 13):  # bytes before each chunk's data (and values before its result)
        payload = torch.full((2 * (lead + n + 8 + 4 * ns),), 0xAA, dtype=torch.uint8)
        scale_at = (2 * (lead + n) + 3) // 4 * 4
        for c in range(2):
            payload[c * (lead + n) + lead:][:n] = data[c].reshape(-1)
            payload[scale_at + 4 * ns * c:][: 4 * ns] = scales[c].reshape(-1).view(torch.uint8)
        table = torch.tensor(
            [[c * (lead + n) + lead, scale_at + 4 * ns * c, rows, in_dim, c * (lead + n) + lead, scale_at + 4 * ns * c,
              c * (lead + n) + lead] for c in range(2)], dtype=torch.int64, device=device)
        starts = torch.tensor([0, ns, 2 * ns], dtype=torch.int64, device=device)
        compact = torch.full_like(payload, 0x55).to(device)
        values = torch.full((2 * (lead + n) + 16,), 7.0, dtype=dtype, device=device)
        hip_ops.unpack_dequant(payload.to(device), table, starts, 2 * ns, compact, values, 128)
        compact, values = compact.cpu(), values.cpu()
        wanted_bytes, wanted_values = torch.full_like(payload, 0x55), torch.full_like(values, 7.0)
        for c in range(2):
            wanted_bytes[c * (lead + n) + lead:][:n] = data[c].reshape(-1)
            wanted_values[c * (lead + n) + lead:][:n] = want[c].reshape(-1)
        wanted_bytes[scale_at:][: 8 * ns] = scales.reshape(-1).view(torch.uint8)
        assert torch.equal(compact, wanted_bytes)
        assert torch.equal(values, wanted_values)
