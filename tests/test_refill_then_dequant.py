"""Every order of unshard steps on a local exchange hands out the bytes that
were exchanged: a refill reads the ranks' rows where they lie and leaves the
gathered rows unwritten, so no finish may read those afterwards.  The launches
are replaced by host loops over the same tables."""

import itertools

import pytest
import torch
import torch.nn as nn

from flex_shard_amd import Fp8BucketedBlockShard, LocalReduceGroup, hip_ops
from flex_shard_amd.blockwise_fp8 import make_blockwise_fp8_weight
from flex_shard_amd.custom_placements import blockwise_quant_bucketed_block_shard as blockwise
from flex_shard_amd.custom_placements import fp8_bucketed_block_shard as fp8
from flex_shard_amd.custom_placements import utils
from flex_shard_amd.placement_contract import PlacementPreparedUnshard
from flex_shard_amd.testing import FakeMesh, make_param_infos, prepare_unshard_on_each_rank


class _ViewShard(Fp8BucketedBlockShard):
    """Hands out (bytes, scales) instead of weights."""

    def _make_quantized_weight_checked(self, qdata, scales, *, orig_dtype, requires_grad):
        return qdata.view(torch.uint8), scales[0]


def _copy_rows(rows, output, descriptor):
    flat = output.view(-1)
    for first, table, _ in descriptor.parts:
        for row, src, nbytes, dst in table.t().tolist():
            flat[dst : dst + nbytes] = rows[first + row].view(-1)[src : src + nbytes]


def _unpack(rows, table, starts, total_tiles, compact, dequant, block):
    source = rows.as_strided((rows.untyped_storage().nbytes() - rows.storage_offset(),), (1,))
    assert int(starts[-1]) == total_tiles
    for src, scale_at, nrows, in_dim, dst, dst_scale, dst_dequant in table.tolist():
        tiles = (-(-nrows // block), -(-in_dim // block))
        nscales = 4 * tiles[0] * tiles[1]
        data, scales = source[src : src + nrows * in_dim], source[scale_at : scale_at + nscales]
        if compact is not None:
            compact[dst : dst + nrows * in_dim] = data
            compact[dst_scale : dst_scale + nscales] = scales
        scale = scales.clone().view(torch.float32).view(tiles)
        scale = scale.repeat_interleave(block, 0)[:nrows].repeat_interleave(block, 1)[:, :in_dim]
        values = data.view(torch.float8_e4m3fn).float().view(nrows, in_dim) * scale
        dequant[dst_dequant : dst_dequant + nrows * in_dim] = values.to(dequant.dtype).view(-1)


@pytest.fixture
def host_launches(monkeypatch):
    def exchange_rows(group, input):
        return [input if r == group.rank() else group.gather_rows[r] for r in range(group.size())]

    monkeypatch.setattr(blockwise, "local_exchange_rows", exchange_rows)
    monkeypatch.setattr(blockwise, "copy_row_segments", _copy_rows)
    monkeypatch.setattr(blockwise, "_require_gpu_rows", lambda *args: None)
    monkeypatch.setattr(fp8, "_require_gpu_rows", lambda *args: None)
    monkeypatch.setattr(hip_ops, "unpack_dequant", _unpack)
    monkeypatch.setattr(hip_ops, "stream_ptr", lambda device: 0)
    pinned = torch.tensor
    monkeypatch.setattr(torch, "tensor", lambda *a, pin_memory=False, **k: pinned(*a, **k))


def _payloads(placement, metadata, world, seed):
    """A row of random FP8 values and scales per rank."""
    gen = torch.Generator().manual_seed(seed)
    rows = []
    for plan in metadata.rank_pack_plans:
        row = torch.zeros(metadata.packed_send_nbytes_per_rank, dtype=torch.uint8)
        row[: plan.scale_byte_offset] = torch.randn(plan.scale_byte_offset, generator=gen).to(torch.float8_e4m3fn).view(torch.uint8)
        nscales = sum(c.scale_numels[0] for c in plan.chunks)
        scales = torch.rand(nscales, generator=gen) + 0.5
        row[plan.scale_byte_offset : plan.scale_byte_offset + 4 * nscales] = scales.view(torch.uint8)
        rows.append(row)
    assert len(rows) == world
    return rows


@pytest.mark.parametrize("shapes,world", [([(256, 136), (130, 257)], 3), ([(128, 128)], 1), ([(3, 130, 136), (300, 40)], 4)])
def test_finishes_after_a_refill_read_what_was_exchanged(host_launches, shapes, world):
    placement = _ViewShard(world_size=world, weight_factory=make_blockwise_fp8_weight)
    named = [(f"w{i}", nn.Parameter(torch.empty(s, device="meta", dtype=torch.bfloat16))) for i, s in enumerate(shapes)]
    infos = make_param_infos(named, placement, FakeMesh(world, 0))
    metadata = placement._quant_metadata_from_infos(infos)

    def prepare(rows, persistent_buffers):
        group = LocalReduceGroup(world, 0)
        group.gather_rows = dict(enumerate(rows))
        stale = torch.full((world * rows[0].numel(),), 0x11, dtype=torch.uint8)  # a recycled gather output
        state = placement._QuantUnshardState(infos, group, None, metadata)
        return PlacementPreparedUnshard(placement, [rows[0], stale], state, True, persistent_buffers)

    def first(rows):
        """The first unshard's finish, from gathered rows."""
        prepared = prepare(rows, None)
        utils.all_gather_rows(prepared.buffers[1], rows[0], prepared.placement_state.pg)
        return placement.finish_prepared_unshard_with_dequant(prepared)

    result, _ = first(_payloads(placement, metadata, world, 0))
    (buffer,) = result.persistent_buffers
    finishes = ("plain", "dequant", "dequant only", "plain, buffer taken away", "dequant, another buffer")
    for seed, order in enumerate(itertools.permutations(finishes, 2), 1):
        rows = _payloads(placement, metadata, world, seed)
        want, want_dequant = first(rows)
        prepared = prepare(rows, [buffer])
        assert placement.run_prepared_unshard(prepared) is None
        for finish in order:
            if "another" in finish:
                prepared.persistent_buffers = [torch.full_like(buffer, 0x22)]
            elif "taken away" in finish:
                prepared.persistent_buffers = None
            if finish.startswith("plain"):
                got, dequant = placement.finish_prepared_unshard(prepared), want_dequant
            else:
                got, dequant = placement.finish_prepared_unshard_with_dequant(prepared, compact=finish == "dequant" or "another" in finish)
            assert all(torch.equal(a, b) for a, b in zip(dequant, want_dequant, strict=True))
            if finish != "dequant only":
                for (data, scale), (want_data, want_scale) in zip(got.full_params, want.full_params, strict=True):
                    assert torch.equal(data, want_data) and torch.equal(scale, want_scale)
        data_end = sum(metadata.rank_qdata_numels)
        assert torch.equal(buffer[:data_end], want.persistent_buffers[0][:data_end])


@pytest.mark.gpu
@pytest.mark.parametrize("dequant_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("world", [1, 3, 8])
def test_dequantizing_finish_of_a_refill_on_the_gpu(device, world, dequant_dtype):
    gen = torch.Generator().manual_seed(world)
    named = [(f"w{i}", nn.Parameter((torch.randn(s, generator=gen) * 0.02).bfloat16().to(device)))
             for i, s in enumerate([(384, 200), (130, 257), (40, 512)])]
    placement = _ViewShard(world_size=world, weight_factory=make_blockwise_fp8_weight)

    def run(persistent_buffers):
        by_rank = prepare_unshard_on_each_rank(placement, named, world)
        prepared, group = by_rank[0], LocalReduceGroup(world, 0)
        group.gather_rows = {r: p.buffers[0] for r, p in enumerate(by_rank)}
        prepared.placement_state.pg = group
        prepared.persistent, prepared.persistent_buffers = True, persistent_buffers
        prepared.buffers[1].fill_(0x11)  # nothing of an earlier exchange is left in the gather output
        placement.run_prepared_unshard(prepared)
        return prepared

    first, want = placement.finish_prepared_unshard_with_dequant(run(None), dequant_dtype=dequant_dtype)
    weights = [(data.clone(), scale.clone()) for data, scale in first.full_params]
    for compact in (True, False, True):
        first.persistent_buffers[0].fill_(0xAB)
        again, got = placement.finish_prepared_unshard_with_dequant(
            run(first.persistent_buffers), dequant_dtype=dequant_dtype, compact=compact
        )
        assert all(torch.equal(a, b) for a, b in zip(got, want, strict=True))
        assert len(again.full_params) == (len(weights) if compact else 0)
        for views, values in zip(first.full_params, weights, strict=True):  # views of the persistent buffer
            assert all(torch.equal(a, b) for a, b in zip(views, values, strict=True))
