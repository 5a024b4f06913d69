"""The exchange of one GPU's ranks without intermediate copies: refills that
read every rank's row where it lies, and reductions that read this rank's own
contribution where it lies."""

import pytest
import torch
import torch.nn as nn

from flex_shard_amd import BucketedBlockShard, Fp8BucketedBlockShard, GradientReduction, LocalReduceGroup, hip_ops
from flex_shard_amd.blockwise_fp8 import make_blockwise_fp8_weight
from flex_shard_amd.flex_shard import begin_bucket_unshard
from flex_shard_amd.testing import FakeMesh, local_rows, make_param_infos

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nrows,nbytes,skew", [(1, 1, 0), (3, 4096, 0), (8, 131073, 5), (32, 65536, 1), (2, 300001, 15)])
def test_row_segments_for_any_alignment(device, nrows, nbytes, skew):
    from flex_shard_amd.custom_placements._copy_kernels import RowCopyDescriptor, copy_row_segments

    rows = [torch.randint(0, 256, (nbytes + skew * r,), dtype=torch.uint8, device=device)[skew * r :] for r in range(nrows)]
    out = torch.full((nrows * nbytes + 64,), 7, dtype=torch.uint8, device=device)
    # rows in reverse, each without its first byte where it has more than one
    cut = 1 if nbytes > 1 else 0
    segments, at = [], 3
    for r in reversed(range(nrows)):
        segments.append((r, cut, nbytes - cut, at))
        at += nbytes - cut
    copy_row_segments(rows, out, RowCopyDescriptor.create(segments, device))
    want = torch.full_like(out, 7)
    for r, src, n, dst in segments:
        want[dst : dst + n] = rows[r][src : src + n]
    assert torch.equal(out, want)


@pytest.mark.parametrize("world", [1, 3, 8])
def test_fp8_refill_equals_the_first_unshard(device, world):
    gen = torch.Generator().manual_seed(world)
    named = [(f"w{i}", nn.Parameter((torch.randn(s, generator=gen) * 0.02).bfloat16().to(device)))
             for i, s in enumerate([(384, 200), (130, 136), (40, 512)])]
    placement = Fp8BucketedBlockShard(world_size=world, weight_factory=make_blockwise_fp8_weight)
    group = LocalReduceGroup(world, 0)
    for other in range(1, world):
        mesh = FakeMesh(world, other)
        infos = make_param_infos(named, placement, mesh)
        shards = [local_rows(p, i) for (_, p), i in zip(named, infos)]
        group.gather_rows[other] = placement.prepare_unshard_bucket(shards, infos, mesh, None).buffers[0].clone()
    mesh = FakeMesh(world, 0, group)
    infos = make_param_infos(named, placement, mesh)
    shards = [local_rows(p, i) for (_, p), i in zip(named, infos)]
    first = begin_bucket_unshard(shards, infos, mesh, None).finish()
    want = [(w.fp8_data.view(torch.uint8).clone(), w.recip_scale.clone()) for w in first.full_params]
    for trial in range(3):
        for t in first.persistent_buffers:
            t.fill_(0xAB)
        if world > 1 and trial == 2:  # the rows moved: the refill reads them where they are now
            group.gather_rows = {r: row.clone() for r, row in group.gather_rows.items()}
        again = begin_bucket_unshard(shards, infos, mesh, None, persistent_buffers=first.persistent_buffers).finish()
        assert again.persistent_buffers[0] is first.persistent_buffers[0]
        for w, (data, scale) in zip(again.full_params, want):
            assert torch.equal(w.fp8_data.view(torch.uint8), data) and torch.equal(w.recip_scale, scale)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("world,rank,seg", [(1, 0, 1000), (2, 1, 4096), (8, 3, 1001), (5, 0, 8)])
def test_own_row_is_read_where_it_lies(device, dtype, world, rank, seg):
    gen = torch.Generator(device=device)
    gen.manual_seed(seg)
    rows = torch.randn((world, world * seg), generator=gen, device=device).to(dtype)
    own = rows[rank].clone()
    for mode, factor in ((hip_ops.REDUCE_SUM, 1.0), (hip_ops.REDUCE_PREMUL, 1 / 3), (hip_ops.REDUCE_POSTDIV, 3.0)):
        want, got = torch.empty(seg, dtype=dtype, device=device), torch.empty(seg, dtype=dtype, device=device)
        hip_ops.reduce_rows(want, rows, rank * seg, mode=mode, factor=factor)
        holed = rows.clone()
        holed[rank] = float("nan")
        hip_ops.reduce_rows(got, holed, rank * seg, mode=mode, factor=factor, own_row=(rank, own))
        assert torch.equal(got, want)


def test_reduction_of_one_rank_needs_no_deposit(device):
    grads = [torch.randn(64, 24, device=device), torch.randn(40, 8, device=device)]
    placement = BucketedBlockShard(dims=(0,), blocks_per_rank=(1,))
    mesh = FakeMesh(1, 0, LocalReduceGroup(1, 0))
    infos = make_param_infos([(f"p{i}", nn.Parameter(g.clone())) for i, g in enumerate(grads)], placement, mesh)
    for info in infos:
        info.reduce_dtype = torch.float32
    for _ in range(2):
        prepared = placement.prepare_reduce_grad(grads, infos, mesh, None)
        shards = placement.reduce_prepared_grad(prepared, GradientReduction()).sharded_grads
        assert all(torch.equal(s.view(g.shape), g) for s, g in zip(shards, grads))
