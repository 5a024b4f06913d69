"""The 128-block unpack walks a chunk as one run of bytes: groups of eight that
reach over a tile's edge, a row's end or both, runs of several workgroups'
pieces, ends shorter than a group, NaN bytes."""

import pytest
import torch

from flex_shard_amd import hip_ops

pytestmark = pytest.mark.gpu
E4M3 = torch.float8_e4m3fn


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,in_dim", [(300, 130), (3, 8), (700, 11), (40, 4099), (2000, 24), (260, 256), (5, 129)])
@pytest.mark.parametrize("lead", [0, 3])  # values ahead of the chunk's
def test_every_kind_of_group(device, rows, in_dim, lead, dtype):
    gen = torch.Generator().manual_seed(rows + in_dim)
    data = torch.randint(0, 256, (rows, in_dim), dtype=torch.uint8, generator=gen)  # NaN bytes among them
    tiles = (-(-rows // 128), -(-in_dim // 128))
    scales = torch.rand(tiles, generator=gen) * 1e-2 + 1e-4
    n, ns = rows * in_dim, tiles[0] * tiles[1]
    want = (data.view(E4M3).float() * scales.repeat_interleave(128, 0)[:rows].repeat_interleave(128, 1)[:, :in_dim]).to(dtype)
    scale_at = (n + 3) // 4 * 4
    source = torch.cat([data.reshape(-1), torch.zeros(scale_at - n, dtype=torch.uint8), scales.reshape(-1).view(torch.uint8)])
    table = torch.tensor([[0, scale_at, rows, in_dim, 0, scale_at, lead]], dtype=torch.int64, device=device)
    starts = torch.tensor([0, ns], dtype=torch.int64, device=device)
    compact = torch.zeros_like(source).to(device)
    values = torch.full((lead + n + 16,), 7.0, dtype=dtype, device=device)
    hip_ops.unpack_dequant(source.to(device), table, starts, ns, compact, values, 128)
    assert torch.equal(compact.cpu(), source)
    got = values.cpu()
    assert (got[:lead] == 7).all() and (got[lead + n :] == 7).all()
    assert torch.equal(torch.nan_to_num(got[lead : lead + n].float(), nan=-1.0), torch.nan_to_num(want.reshape(-1).float(), nan=-1.0))
    only = torch.full_like(values, 7.0)  # the values without the compact bytes, and the reverse
    hip_ops.unpack_dequant(source.to(device), table, starts, ns, None, only, 128)
    assert torch.equal(only.cpu().view(torch.uint8), got.view(torch.uint8))
    again = torch.zeros_like(compact)
    hip_ops.unpack_dequant(source.to(device), table, starts, ns, again, None, 128)
    assert torch.equal(again, compact)
