"""The cached layout behind a finished FP8 unshard against the general
split-and-view path, over the forms it accepts: views of the same bytes, with
the same shapes and strides, and the same refusals."""

import pytest
import torch
import torch.nn as nn

from flex_shard_amd import Fp8BucketedBlockShard
from flex_shard_amd.testing import FakeMesh, make_param_infos


def _factory(fp8_data, recip_scale, block_size, *, orig_dtype, requires_grad):
    assert block_size == 128 and orig_dtype == torch.bfloat16
    fp8_data.recip_scale = recip_scale
    return fp8_data


class _ColumnMajorScales(Fp8BucketedBlockShard):
    def _param_scale_view(self, scale_index, scale, matrix_shape):
        return super()._param_scale_view(scale_index, scale, matrix_shape).t()


def _state(shapes, world, cls=Fp8BucketedBlockShard):
    placement = cls(world_size=world, weight_factory=_factory)
    named = [(f"w{i}", nn.Parameter(torch.empty(s, device="meta", dtype=torch.bfloat16))) for i, s in enumerate(shapes)]
    infos = make_param_infos(named, placement, FakeMesh(world, 0))
    state = placement._QuantUnshardState(infos, None, None, placement._quant_metadata_from_infos(infos))
    _, scale_start, groups = placement._compact_sizes(state.metadata)
    return placement, state, scale_start + sum(groups)


def _describe(views):
    return [(t.data_ptr(), t.dtype, t.shape, t.stride()) for v in views for t in (v, v.recip_scale)]


@pytest.mark.parametrize("offset", [0, 64])
@pytest.mark.parametrize("cls", [Fp8BucketedBlockShard, _ColumnMajorScales])
@pytest.mark.parametrize(
    "shapes,world",
    [([(128, 128)], 1), ([(1, 8), (130, 257), (128, 1)], 2), ([(3, 130, 136), (300, 40)], 3), ([(256, 512)] * 5, 8)],
)
def test_cached_views_are_those_of_the_general_path(monkeypatch, shapes, world, cls, offset):
    placement, state, nbytes = _state(shapes, world, cls)
    compact = torch.zeros(offset + nbytes, dtype=torch.uint8)[offset:]
    cached = _describe(placement._full_params_from_compact(state, compact))
    again = _describe(placement._full_params_from_compact(state, compact))
    assert (placement._full_param_plan(state) is None) == (cls is _ColumnMajorScales)
    monkeypatch.setattr(placement, "_full_param_plan", lambda state: None)
    assert cached == again == _describe(placement._full_params_from_compact(state, compact))


@pytest.mark.parametrize("extra", [-4, 4])
def test_buffer_of_another_size_is_refused(extra):
    placement, state, nbytes = _state([(130, 136), (64, 128)], 2)
    placement._full_params_from_compact(state, torch.zeros(nbytes, dtype=torch.uint8))
    with pytest.raises(RuntimeError, match="split_with_sizes"):
        placement._full_params_from_compact(state, torch.zeros(nbytes + extra, dtype=torch.uint8))


def test_other_infos_of_the_same_layout_are_looked_at_again():
    placement, state, nbytes = _state([(128, 256), (128, 256)], 2)
    compact = torch.zeros(nbytes, dtype=torch.uint8)
    first = _describe(placement._full_params_from_compact(state, compact))
    state.infos = list(state.infos)
    assert _describe(placement._full_params_from_compact(state, compact)) == first
    state.infos = state.infos[:1]
    with pytest.raises(RuntimeError, match="split_with_sizes"):
        placement._full_params_from_compact(state, compact)
