"""A local exchange of more ranks than one launch carries row addresses for
stays on the copy kernel: a launch for every 32 rows, not a copy per row."""

import pytest
import torch

from flex_shard_amd import LocalReduceGroup, hip_ops
from flex_shard_amd._native import MAX_COPY_ROWS
from flex_shard_amd.custom_placements import _copy_kernels, utils


@pytest.mark.parametrize("nrows", [1, MAX_COPY_ROWS, MAX_COPY_ROWS + 1, 3 * MAX_COPY_ROWS + 5])
def test_descriptor_parts_cover_every_row_once(monkeypatch, nrows):
    launches = []
    monkeypatch.setattr(_copy_kernels, "_upload_i64", lambda values, device: (torch.tensor(values), torch.tensor(values)))
    monkeypatch.setattr(hip_ops, "copy_row_segments", lambda rows, out, table, longest: launches.append((rows, table, longest)))
    segments = [(r, 3 * r, 1000 + r, 2000 * r) for r in reversed(range(nrows))] + [(0, 0, 0, 0)]
    _copy_kernels.copy_row_segments(list(range(nrows)), None, _copy_kernels.RowCopyDescriptor.create(segments, None, max_piece_nbytes=600))
    assert len(launches) == -(-nrows // MAX_COPY_ROWS)
    copied = {}
    for rows, table, longest in launches:
        assert len(rows) <= MAX_COPY_ROWS and longest == table[2].max()
        for row, src, nbytes, dst in table.t().tolist():
            copied.setdefault(rows[row], []).append((src, nbytes, dst))
    assert copied == {r: [(3 * r, 600, 2000 * r), (3 * r + 600, 400 + r, 2000 * r + 600)] for r in range(nrows)}


@pytest.mark.gpu
@pytest.mark.parametrize("world,rank", [(MAX_COPY_ROWS, 3), (MAX_COPY_ROWS + 1, MAX_COPY_ROWS), (70, 5)])
def test_all_gather_of_many_ranks(device, monkeypatch, world, rank):
    rows = [torch.randint(0, 256, (50_003,), dtype=torch.uint8, device=device) for _ in range(world)]
    group = LocalReduceGroup(world, rank)
    group.gather_rows = {r: row for r, row in enumerate(rows) if r != rank}
    launches = []
    launch = hip_ops.copy_row_segments
    monkeypatch.setattr(hip_ops, "copy_row_segments", lambda *args: (launches.append(len(args[0])), launch(*args)))
    out = torch.zeros(world * 50_003, dtype=torch.uint8, device=device)
    utils.all_gather_rows(out, rows[rank], group)
    assert torch.equal(out, torch.cat(rows)) and sum(launches) == world and len(launches) == -(-world // MAX_COPY_ROWS)
