"""A local reduction that was refused (a contribution missing, an output of the
wrong size) and is called again reads this rank's contribution, never a row
that nobody wrote.  The launch is replaced by a host loop."""

import pytest
import torch

from flex_shard_amd import GradientReduction, LocalReduceGroup, hip_ops
from flex_shard_amd.custom_placements import utils


class _OnGpu:
    """A device that says it is a GPU."""

    type = "cuda"

    def __eq__(self, other):
        return isinstance(other, _OnGpu)


class _GpuLike(torch.Tensor):
    device = property(lambda self: _OnGpu())


def _fold(out, contributions, column_offset, *, mode, factor, own_row=None):
    rows = contributions.as_subclass(torch.Tensor).clone()
    if own_row is not None:
        rows[own_row[0]] = own_row[1].as_subclass(torch.Tensor)
    out.copy_(rows[:, column_offset : column_offset + out.numel()].sum(0) * (factor if mode == hip_ops.REDUCE_PREMUL else 1.0))


def _setup(monkeypatch, world, rank, seg):
    monkeypatch.setattr(hip_ops, "reduce_rows", _fold)
    gen = torch.Generator().manual_seed(world * 10 + rank)
    sent = torch.randint(-8, 8, (world, world * seg), generator=gen).float()
    group = LocalReduceGroup(world, rank)
    group.contributions = torch.full((world, world * seg), float("nan")).as_subclass(_GpuLike)
    return sent, group, torch.empty(seg).as_subclass(_GpuLike), sent[rank].clone().as_subclass(_GpuLike)


@pytest.mark.parametrize("world,rank", [(2, 0), (3, 1), (8, 7)])
def test_contribution_deposited_after_the_refusal(monkeypatch, world, rank):
    seg = 5
    sent, group, out, own = _setup(monkeypatch, world, rank, seg)
    others = [r for r in range(world) if r != rank]
    for step in range(2):  # and again with what the first reduction left behind
        for r in others[1:]:
            group.deposit(r, sent[r])
        with pytest.raises(ValueError, match=f"missing the contributions of ranks \\[{others[0]}\\]"):
            utils.reduce_scatter_grads(out, own, GradientReduction(op="sum"), group)
        group.deposit(others[0], sent[others[0]])
        utils.reduce_scatter_grads(out, own, GradientReduction(op="sum"), group)
        assert torch.equal(out.as_subclass(torch.Tensor), sent.sum(0)[rank * seg : (rank + 1) * seg])
        assert not group.deposited
        sent.mul_(2.0)
        own = sent[rank].clone().as_subclass(_GpuLike)


@pytest.mark.parametrize("world,rank", [(1, 0), (3, 1)])
def test_output_of_the_wrong_size(monkeypatch, world, rank):
    seg = 6
    sent, group, out, own = _setup(monkeypatch, world, rank, seg)
    for r in range(world):
        if r != rank:
            group.deposit(r, sent[r])
    with pytest.raises(ValueError, match="Expected contributions of shape"):
        utils.reduce_scatter_grads(out[1:], own, GradientReduction(op="sum"), group)
    utils.reduce_scatter_grads(out, own, GradientReduction(op="sum"), group)
    assert torch.equal(out.as_subclass(torch.Tensor), sent.sum(0)[rank * seg : (rank + 1) * seg])
