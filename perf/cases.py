"""The work whose speed is measured: what a training program has this package
do on one GPU, through its public entry points, from single small calls to
whole training steps.

A case is a dict of plain values; ``path`` says which entry points it takes:

``unshard_fp8``    one rank's FP8 bucket unshard: quantize + pack the local
                   shards, exchange, unpack into the persistent buffers (or
                   unpack + dequantize in one pass)
``unshard_dense``  the same bucket step without quantization (cast + gather)
``reduce_grads``   a bucket's gradient path: microbatch accumulation in fp32 or
                   the casting copy-in, then the fixed-order reduction
``linear``         the blockwise FP8 linear on a gathered weight, forward alone
                   or forward + backward
``muon``           one optimizer step on the whole matrices a rank owns
``train_block``    forward + backward of blocks of FP8 projections under the
                   bucket runtime's hooks (unshard, linears, reshard, reduce)

Shapes are written as text, "rows x cols" joined by commas.  The exchange of a
mesh of several ranks is the package's one-GPU stand-in (``LocalReduceGroup``):
the other ranks' rows and contributions are inputs like any other.
"""

from __future__ import annotations

import math

import torch
import torch.nn as nn

from flex_shard_amd import BucketedBlockShard, Fp8BucketedBlockShard, GradientReduction, LocalReduceGroup, hip_ops
from flex_shard_amd.blockwise_fp8 import (
    convert_to_flex_shard_float8_blockwise_linear,
    make_blockwise_fp8_weight,
    prequantized_linear,
)
from flex_shard_amd.blockwise_fp8.fp8_blockwise_linear import shared_activation_quantizer
from flex_shard_amd.dist_muon import OwnedMuon
from flex_shard_amd.flex_shard import BucketCommContext, BucketRuntime, begin_bucket_unshard
from flex_shard_amd.testing import FakeMesh, local_rows, make_param_infos

# q, k, v, o, gate, up, down of a Llama-3-8B layer: the benchmark's bucket
LAYER = "4096x4096,1024x4096,1024x4096,4096x4096,14336x4096,14336x4096,4096x14336"
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def listed() -> list[dict]:
    return [
        # A small bucket (two 2048 x 2048 weights, two ranks): what a step of a
        # small model or a bucket of few parameters costs; latency and launches.
        {"name": "unshard_fp8_small", "path": "unshard_fp8", "shapes": "2048x2048,2048x2048", "world": 2, "rank": 0,
         "master": "bf16", "dequant": False},
        # The benchmark's layer bucket on the first of eight ranks, twice per
        # layer and step in training (forward and backward).
        {"name": "unshard_fp8_layer", "path": "unshard_fp8", "shapes": LAYER, "world": 8, "rank": 0, "master": "bf16",
         "dequant": False},
        # fp32 masters, three ranks, rows that are not whole blocks and a
        # width that is not a multiple of 16, bf16 weights wanted as well (a
        # consumer without an FP8 product): an odd model's bucket.
        {"name": "unshard_fp8_ragged_dequant", "path": "unshard_fp8", "shapes": "3000x1544,1000x1544,1544x3000,777x1000",
         "world": 3, "rank": 1, "master": "fp32", "dequant": True},
        # The layer bucket without quantization: fp32 masters gathered as bf16.
        {"name": "unshard_dense_layer", "path": "unshard_dense", "shapes": LAYER, "world": 8, "rank": 3,
         "master": "fp32"},
        # Four microbatches accumulated in fp32 in the flat gradient bucket of
        # the layer, then reduced over eight ranks.
        {"name": "reduce_grads_layer", "path": "reduce_grads", "shapes": LAYER, "world": 8, "rank": 0,
         "microbatches": 4},
        # Separate bf16 gradients of an odd model's bucket, widened by the
        # copy-in, reduced over three ranks.
        {"name": "reduce_grads_ragged", "path": "reduce_grads", "shapes": "3000x1544,1000x1544,1544x3000,777x1000",
         "world": 3, "rank": 2, "microbatches": 0},
        # Few tokens through a wide projection, forward only: sampling from or
        # probing the model between training steps.
        {"name": "linear_few_tokens", "path": "linear", "tokens": 48, "shape": "14336x4096", "backward": False,
         "bias": False},
        # A training microbatch of an odd length (packed sequences) through a
        # mid-sized projection with a bias.
        {"name": "linear_odd_microbatch", "path": "linear", "tokens": 1000, "shape": "5120x2048", "backward": True,
         "bias": True},
        # The optimizer step of a small model: many small matrices, some of odd
        # shapes.
        {"name": "muon_small_matrices", "path": "muon",
         "groups": "8*768x768,4*3072x768,4*768x3072,2*1000x520,2*300x700", "master": "bf16"},
        # One rank's share of a layer's projections kept as fp32 masters.
        {"name": "muon_layer_fp32", "path": "muon", "groups": "2*4096x4096,2*1024x4096,1*14336x4096",
         "master": "fp32"},
        # The benchmark's 48 whole matrices of one rank.
        {"name": "muon_48_matrices", "path": "muon", "groups": "24*7168x2048,24*2048x2048", "master": "bf16"},
        # One block of the seven projections at 8192 tokens, forward and
        # backward under the runtime's hooks, first of eight ranks.
        {"name": "train_block_8192_tokens", "path": "train_block", "dim": 4096, "kv_dim": 1024, "hidden": 14336,
         "tokens": 8192, "world": 8, "blocks": 1, "master": "bf16"},
    ]


def _log_int(rng, low: int, high: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _dim(rng, low: int, high: int) -> int:
    """A matrix dimension: mostly multiples of 128 (as models have them), some
    of 8, a few of any size."""
    value = _log_int(rng, low, high)
    step = rng.choice((128, 128, 128, 64, 8, 1))
    return min(high, max(step, value // step * step, 1))


def draw(rng) -> dict:
    path = rng.choice(("unshard_fp8", "unshard_fp8", "unshard_dense", "reduce_grads", "reduce_grads", "linear", "linear",
                       "linear", "muon", "muon", "muon", "train_block"))
    if path in ("unshard_fp8", "unshard_dense", "reduce_grads"):
        budget = _log_int(rng, 1 << 20, 218_000_000)  # elements of the bucket
        count = rng.randint(1, 8)
        base = _dim(rng, 256, 3584)
        shapes = []
        for _ in range(count):
            # a dense bucket aligns its parameters to a common multiple of
            # their widths, so these are multiples of one another in a model
            cols = _dim(rng, 256, 14336) if path == "unshard_fp8" else base * rng.choice((1, 1, 2, 4))
            rows = max(1, min(28672, int(budget / count / cols * rng.uniform(0.4, 1.2))))
            if rng.random() < 0.7:
                rows = max(128, rows // 128 * 128)
            shapes.append(f"{rows}x{cols}")
        world = rng.choice((1, 2, 3, 4, 8, 8))
        case = {"path": path, "shapes": ",".join(shapes), "world": world, "rank": rng.randrange(world)}
        if path == "unshard_fp8":
            case.update(master=rng.choice(("bf16", "bf16", "fp32")), dequant=rng.random() < 0.4)
        elif path == "unshard_dense":
            case.update(master=rng.choice(("bf16", "fp32")))
        else:
            case.update(microbatches=rng.choice((0, 0, 1, 2, 4)))
        return case
    if path == "linear":
        return {"path": path, "tokens": _log_int(rng, 1, 8192), "shape": f"{_dim(rng, 512, 14336)}x{_dim(rng, 512, 14336)}",
                "backward": rng.random() < 0.6, "bias": rng.random() < 0.3}
    if path == "muon":
        target = math.exp(rng.uniform(math.log(2e10), math.log(1.5e13)))  # flops of the step
        groups = []
        for _ in range(rng.randint(1, 3)):
            rows, cols = _dim(rng, 256, 7168), _dim(rng, 256, 7168)
            if rng.random() < 0.3:
                rows = cols
            s, l = min(rows, cols), max(rows, cols)
            count = max(1, min(16, int(target / 3 / (10 * s * s * (2 * l + s)))))
            groups.append(f"{count}*{rows}x{cols}")
        return {"path": path, "groups": ",".join(groups), "master": rng.choice(("bf16", "bf16", "fp32"))}
    dim = rng.choice((1024, 1536, 2048, 2560, 4096))
    return {"path": path, "dim": dim, "kv_dim": dim // rng.choice((1, 2, 4)), "hidden": dim * rng.choice((2, 3, 4)) // 2,
            "tokens": _log_int(rng, 256, 8192), "world": rng.choice((1, 2, 4, 8)), "blocks": rng.randint(1, 2),
            "master": rng.choice(("bf16", "fp32"))}


# ---------------------------------------------------------------- making inputs
def _shapes(text: str) -> list[tuple[int, int]]:
    return [tuple(int(n) for n in part.split("x")) for part in text.split(",")]


def _groups(text: str) -> list[tuple[int, int, int]]:
    out = []
    for part in text.split(","):
        count, shape = part.split("*")
        out.append((int(count), *(int(n) for n in shape.split("x"))))
    return out


class _Random:
    """Normal tensors on the GPU, one after the other from one seed."""

    def __init__(self, seed: int) -> None:
        self.device = torch.device("cuda:0")
        self.gen = torch.Generator(device=self.device)
        self.gen.manual_seed(seed)

    def normal(self, shape, std: float, dtype=torch.bfloat16) -> torch.Tensor:
        out = torch.empty(shape, dtype=torch.float32, device=self.device)
        out.normal_(0.0, std, generator=self.gen)
        return out if dtype == torch.float32 else out.to(dtype)


def _bucket(case: dict, placement, mesh, master: torch.dtype, rng: _Random):
    """This rank's ParamInfos and its shards as views of one flat storage."""
    named = [(f"p{i}", nn.Parameter(torch.empty(s, device="meta", dtype=master)))
             for i, s in enumerate(_shapes(case["shapes"]))]
    infos = make_param_infos(named, placement, mesh)
    for info in infos:
        info.param_dtype = torch.bfloat16
        info.reduce_dtype = torch.float32
    local = infos[0].bucket_layout.local_numel
    size = master.itemsize
    storage = torch.zeros(local, dtype=master, device=rng.device)
    shards = []
    for info in infos:
        start = info.byte_offset // size
        view = storage[start : start + info.local_numel]
        view.copy_(rng.normal((info.local_numel,), 0.02, master))
        shards.append(view.view(info.local_shape))
    return infos, storage, shards


def _prepare_unshard(case: dict, rng: _Random) -> dict:
    world, rank, master = case["world"], case["rank"], DTYPES[case["master"]]
    if case["path"] == "unshard_fp8":
        placement = Fp8BucketedBlockShard(world_size=world, weight_factory=make_blockwise_fp8_weight)
    else:
        placement = BucketedBlockShard(dims=(0,), blocks_per_rank=(1,) * world)
    group = LocalReduceGroup(world, rank)
    for other in range(world):  # what the other ranks send
        if other != rank:
            mesh = FakeMesh(world, other)
            infos, _, shards = _bucket(case, placement, mesh, master, rng)
            group.gather_rows[other] = placement.prepare_unshard_bucket(shards, infos, mesh, None).buffers[0].clone()
    mesh = FakeMesh(world, rank, group)
    infos, storage, shards = _bucket(case, placement, mesh, master, rng)
    state = {"path": case["path"], "placement": placement, "mesh": mesh, "infos": infos, "storage": storage,
             "shards": shards, "buffers": None, "full": None, "dequant": None}
    if case.get("dequant"):
        state["dequant"] = torch.empty(sum(i.global_numel for i in infos), dtype=torch.bfloat16, device=rng.device)
    return state


def _prepare_reduce(case: dict, rng: _Random) -> dict:
    world, rank = case["world"], case["rank"]
    placement = BucketedBlockShard(dims=(0,), blocks_per_rank=(1,) * world)
    group = LocalReduceGroup(world, rank)
    mesh = FakeMesh(world, rank, group)
    shapes = _shapes(case["shapes"])
    named = [(f"p{i}", nn.Parameter(torch.empty(s, device="meta", dtype=torch.bfloat16))) for i, s in enumerate(shapes)]
    infos = make_param_infos(named, placement, mesh)
    for info in infos:
        info.reduce_dtype = torch.float32
    layout = infos[0].bucket_layout
    send_numel = world * max(layout.rank_numels)
    rows = group.allocate(send_numel, torch.float32, rng.device)
    for other in range(world):
        if other != rank:
            rows[other].normal_(0.0, 1e-3, generator=rng.gen)
    state = {"path": case["path"], "placement": placement, "mesh": mesh, "infos": infos, "group": group,
             "reduction": GradientReduction(), "others": [r for r in range(world) if r != rank]}
    if case["microbatches"]:
        # The gradients of a microbatch in the bucket's layout, and the fp32
        # bucket they accumulate in (its parameters are views).
        state["micro"] = [torch.zeros(layout.global_numel, dtype=torch.bfloat16, device=rng.device)
                          for _ in range(case["microbatches"])]
        spans = []
        for info in infos:
            start = layout.param_layouts[info.fqn].param_offset
            spans.append((start, start + info.global_numel, info.global_shape))
        for flat in state["micro"]:
            for start, stop, shape in spans:
                flat[start:stop] = rng.normal((stop - start,), 1e-3)
        state["acc"] = torch.zeros(layout.global_numel, dtype=torch.float32, device=rng.device)
        state["grads"] = [state["acc"][start:stop].view(shape) for start, stop, shape in spans]
    else:
        state["micro"], state["acc"] = [], None
        state["grads"] = [rng.normal(s, 1e-3) for s in shapes]
    return state


def _prepare_linear(case: dict, rng: _Random) -> dict:
    (out_dim, in_dim), tokens = _shapes(case["shape"])[0], case["tokens"]
    # the gathered weight as an unshard on one rank leaves it
    placement = Fp8BucketedBlockShard(world_size=1, weight_factory=make_blockwise_fp8_weight)
    mesh = FakeMesh(1, 0, LocalReduceGroup(1, 0))
    weight = nn.Parameter(rng.normal((out_dim, in_dim), 0.02))
    infos = make_param_infos([("w", weight)], placement, mesh)
    gathered = begin_bucket_unshard([weight.detach()], infos, mesh, None).finish().full_params[0]
    x = rng.normal((tokens, in_dim), 1.0)
    state = {"path": case["path"], "backward": case["backward"], "x": x, "weight": gathered,
             "bias": rng.normal((out_dim,), 0.02) if case["bias"] else None}
    if case["backward"]:
        state["x"] = x.requires_grad_()
        state["weight"] = nn.Parameter(gathered)
        if case["bias"]:
            state["bias"].requires_grad_()
        state["grad_out"] = rng.normal((tokens, out_dim), 0.01)
    return state


def _prepare_muon(case: dict, rng: _Random) -> dict:
    dtype = DTYPES[case["master"]]
    storages, params, grads = [], [], []
    for count, rows, cols in _groups(case["groups"]):
        # the matrices of a bucket lie in one storage, their gradients anywhere
        storages.append(rng.normal((count, rows, cols), 0.02, dtype))
        params += storages[-1].unbind(0)
        grads += [rng.normal((rows, cols), 1.0, dtype) for _ in range(count)]
    return {"path": case["path"], "optimizer": OwnedMuon(params, lr=0.02), "storages": storages, "grads": grads}


class _Projections(nn.Module):
    """q, k, v, o and gate, up, down of one block joined by elementwise
    operations (attention itself and the norms belong to the model)."""

    def __init__(self, dim: int, kv_dim: int, hidden: int) -> None:
        super().__init__()
        for name, out_dim, in_dim in _projections(dim, kv_dim, hidden):
            setattr(self, name, nn.Linear(in_dim, out_dim, bias=False, device="meta"))
        self.repeat = dim // (2 * kv_dim) if dim >= 2 * kv_dim else 0

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        k, v = self.k(x), self.v(x)
        kv = torch.cat([k, v], dim=-1).repeat(1, self.repeat) if self.repeat else k + v
        h = self.o(self.q(x) + kv)
        return self.down(self.gate(h) * self.up(h))


def _projections(dim: int, kv_dim: int, hidden: int) -> list[tuple[str, int, int]]:
    return [("q", dim, dim), ("k", kv_dim, dim), ("v", kv_dim, dim), ("o", dim, dim), ("gate", hidden, dim),
            ("up", hidden, dim), ("down", dim, hidden)]


def _prepare_train(case: dict, rng: _Random) -> dict:
    world, master = case["world"], DTYPES[case["master"]]
    sizes = (case["dim"], case["kv_dim"], case["hidden"])
    context = BucketCommContext.create(rng.device)
    blocks, runtimes, groups = [], [], []
    for _ in range(case["blocks"]):
        block = _Projections(*sizes)
        for name, out_dim, in_dim in _projections(*sizes):
            getattr(block, name).weight = nn.Parameter(rng.normal((out_dim, in_dim), 0.02, master))
        convert_to_flex_shard_float8_blockwise_linear(block)
        fqns = [f"{name}.weight" for name, _, _ in _projections(*sizes)]
        named = [(fqn, block.get_parameter(fqn)) for fqn in fqns]
        placement = Fp8BucketedBlockShard(world_size=world, weight_factory=make_blockwise_fp8_weight)
        group = LocalReduceGroup(world, 0)
        for other in range(1, world):
            mesh = FakeMesh(world, other)
            infos = make_param_infos(named, placement, mesh)
            for info in infos:
                info.param_dtype = torch.bfloat16
            shards = [local_rows(p, i) for (_, p), i in zip(named, infos)]
            group.gather_rows[other] = placement.prepare_unshard_bucket(shards, infos, mesh, None).buffers[0].clone()
        runtime = BucketRuntime.shard_module_params(block, fqns, placement, FakeMesh(world, 0, group), context,
                                                    GradientReduction())
        for info in runtime.infos:
            info.param_dtype = torch.bfloat16
        widest = max(runtime.infos[0].bucket_layout.rank_numels)
        rows = group.allocate(world * widest, torch.float32, rng.device)
        for other in range(1, world):
            rows[other].normal_(0.0, 1e-3, generator=rng.gen)
        blocks.append(block)
        runtimes.append(runtime)
        groups.append(group)
    for index, (block, runtime) in enumerate(zip(blocks, runtimes)):
        runtime.install_hooks(
            block,
            forward_prefetch=runtimes[index + 1] if index + 1 < len(runtimes) else None,
            backward_prefetch=runtimes[index - 1] if index > 0 else None,
        )
    return {"path": case["path"], "model": nn.Sequential(*blocks), "runtimes": runtimes, "groups": groups,
            "context": context, "x": rng.normal((case["tokens"], case["dim"]), 1.0).requires_grad_(),
            "grad_out": rng.normal((case["tokens"], case["dim"]), 0.01)}


def prepare(case: dict, seed: int) -> dict:
    rng = _Random(seed)
    path = case["path"]
    if path in ("unshard_fp8", "unshard_dense"):
        return _prepare_unshard(case, rng)
    return {"reduce_grads": _prepare_reduce, "linear": _prepare_linear, "muon": _prepare_muon,
            "train_block": _prepare_train}[path](case, rng)


# --------------------------------------------------------------------- one pass
def _fp8_outputs(weights) -> list[torch.Tensor]:
    return [t for w in weights for t in (w.fp8_data.view(torch.uint8), w.recip_scale)]


def _run_unshard(state: dict):
    if state["dequant"] is not None:
        placement = state["placement"]
        prepared = placement.prepare_unshard_bucket(state["shards"], state["infos"], state["mesh"], None)
        placement.run_prepared_unshard(prepared)
        result, weights = placement.finish_prepared_unshard_with_dequant(prepared, dequant_out=state["dequant"])
        return _fp8_outputs(result.full_params) + weights
    # The first unshard creates the persistent buffers, later ones refill them.
    handle = begin_bucket_unshard(state["shards"], state["infos"], state["mesh"], None,
                                  persistent_buffers=state["buffers"])
    result = handle.finish()
    if state["path"] == "unshard_fp8":
        state["buffers"] = result.persistent_buffers
        return _fp8_outputs(result.full_params)
    if state["buffers"] is None:
        state["buffers"], state["full"] = result.persistent_buffers, result.full_params
    return list(state["full"])


def _run_reduce(state: dict):
    for index, micro in enumerate(state["micro"]):
        hip_ops.accumulate_grad(state["acc"], micro, overwrite=index == 0)
    placement, group = state["placement"], state["group"]
    group.mark_deposited(*state["others"])
    prepared = placement.prepare_reduce_grad(state["grads"], state["infos"], state["mesh"], None)
    result = placement.reduce_prepared_grad(prepared, state["reduction"])
    return [prepared.buffers[0], *result.sharded_grads]


def _run_linear(state: dict):
    # A step's activations are new: nothing quantized in the step before serves this one.
    shared_activation_quantizer.clear()
    x, weight, bias = state["x"], state["weight"], state["bias"]
    if not state["backward"]:
        with torch.no_grad():
            return prequantized_linear(x, weight, bias)
    out = prequantized_linear(x, weight, bias)
    wanted = [x, weight] if bias is None else [x, weight, bias]
    return [out.detach(), *torch.autograd.grad(out, wanted, state["grad_out"])]


def _run_muon(state: dict):
    optimizer = state["optimizer"]
    optimizer.step(state["grads"])
    return [*state["storages"], *optimizer.momentum_buffers]


def _run_train(state: dict):
    shared_activation_quantizer.clear()
    for group in state["groups"]:
        group.mark_deposited(*range(1, group.size()))
    x = state["x"]
    x.grad = None
    for runtime in state["runtimes"]:
        for p in runtime.sharded_params:
            p.grad = None
    out = state["model"](x)
    out.backward(state["grad_out"])
    state["context"].wait_and_clear_reduce_grad_states()
    return [out.detach(), x.grad, *[p.grad for r in state["runtimes"] for p in r.sharded_params]]


def run(state: dict):
    path = state["path"]
    if path in ("unshard_fp8", "unshard_dense"):
        return _run_unshard(state)
    return {"reduce_grads": _run_reduce, "linear": _run_linear, "muon": _run_muon, "train_block": _run_train}[path](state)


# ------------------------------------------------------------- what a pass needs
def work(case: dict) -> dict:
    path = case["path"]
    if path in ("unshard_fp8", "unshard_dense", "reduce_grads"):
        shapes, world = _shapes(case["shapes"]), case["world"]
        total = sum(r * c for r, c in shapes)
        share = total / world
        if path == "reduce_grads":
            # gradients read, the reduce-scatter input (or the accumulated bucket) and the reduced shard
            # written, the other ranks' contributions to this shard read
            grads = 2 * total * max(1, case["microbatches"])
            return {"bytes": int(grads + 4 * total + 4 * share * (world - 1) + 4 * share),
                    "flops": int(total * max(0, case["microbatches"] - 1) + share * world)}
        size = DTYPES[case["master"]].itemsize
        if path == "unshard_dense":
            return {"bytes": int(size * share + 2 * (total - share) + 2 * total), "flops": 0}
        scales = sum(-(-r // 128) * -(-c // 128) for r, c in shapes)
        nbytes = size * share + (total - share) + total + 8 * scales + (2 * total if case["dequant"] else 0)
        return {"bytes": int(nbytes), "flops": int(2 * share)}
    if path == "linear":
        (n, k), m = _shapes(case["shape"])[0], case["tokens"]
        nbytes = 2 * m * k + n * k + 4 * (-(-n // 128)) * (-(-k // 128)) + 2 * m * n
        if case["backward"]:
            nbytes += 2 * m * n + 2 * m * k + 2 * n * k
        return {"bytes": nbytes, "flops": 2 * m * n * k * (3 if case["backward"] else 1)}
    if path == "muon":
        size = DTYPES[case["master"]].itemsize
        nbytes = flops = 0
        for count, rows, cols in _groups(case["groups"]):
            s, l = min(rows, cols), max(rows, cols)
            nbytes += count * rows * cols * 5 * size
            flops += count * 5 * (s * s * (l + s) + 2 * s * s * l)  # two of the three products are symmetric
        return {"bytes": nbytes, "flops": flops}
    layers = [(o, i) for _, o, i in _projections(case["dim"], case["kv_dim"], case["hidden"])] * case["blocks"]
    m, world, size = case["tokens"], case["world"], DTYPES[case["master"]].itemsize
    total = sum(o * i for o, i in layers)
    # shards read for both unshards, the other ranks' bytes and contributions, gradients of the shards; x, out and their gradients
    nbytes = 2 * (size * total / world + total) + 4 * total + size * total / world + 8 * m * case["dim"]
    return {"bytes": int(nbytes), "flops": 6 * m * total}


def tolerance(case: dict):
    path = case["path"]
    if path in ("unshard_fp8", "unshard_dense"):
        return "exact"  # bytes, scales, casts and dequantized values are defined to the bit
    if path == "reduce_grads":
        return {"rel": 2.5e-7}  # fp32 sums: 6e-8 from the same sums in 64 bits
    if path == "linear":
        # 2.3e-4 (largest 0.025) from the same products summed in 64 bits: bf16 results on the other side of a rounding
        return {"rel": 1e-3, "max": 0.1}
    if path == "muon":
        # 8e-4 (largest 0.025) from the iteration with fp32 or 64-bit products rounded at the same points: the
        # orthogonalized matrices differ by 6e-3, the parameters they update by that times the step
        return {"rel": 3e-3, "max": 0.1}
    # A value on the other side of a bf16 rounding changes the scale or the FP8 rounding of its run in the next
    # linear: 0.04 (one block) and 0.11 (two) from the same step with its products summed in 64 bits.
    return {"rel": 0.16 if case["blocks"] == 1 else 0.4}
