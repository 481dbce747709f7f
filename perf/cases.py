"""The KV-block transfers a serving program makes, as measurable cases.

A case describes one call: which direction, the cache geometry (layers, K/V
heads, head size, tokens per block, bytes per element, one latent half or K
and V), how many blocks move, how their ids are spread, and the options of the
call.  The bytes moved are copied, never computed, so every output is compared
exactly.

Kinds:
  save     device to host (``transfer_kv_blocks``): blocks of a finished or
           evicted request go to the pinned host cache
  load     host to device: a prefix hit comes back before its prefill
  stream   host to device layer by layer (``transfer_kv_blocks_layerwise``):
           the prefill of layer l waits for layer l only
  gather   device cache to one contiguous device buffer (RDMA, peer GPUs,
           files), ``gather_kv_blocks``
  scatter  the way back, ``scatter_kv_blocks``
"""
import math

import torch

from flexkv_amd import c_ext
from flexkv_amd.storage.allocator import pinned_empty

DEVICE = "cuda:0"
MIB = 1 << 20

# (layers, K/V heads, head size, one latent half): the Llama-3-8B cache, a
# Llama-3-70B TP-8 shard, the DeepSeek MLA latent and the 4-layer CPU-plumbing
# shape of the benchmark configurations.
LLAMA8B = dict(layers=32, heads=8, dim=128, mla=False)
LLAMA70B_TP8 = dict(layers=80, heads=1, dim=128, mla=False)
MLA = dict(layers=61, heads=1, dim=576, mla=True)
SMALL = dict(layers=4, heads=8, dim=128, mla=False)


def _case(name, kind, model, blocks, tokens=16, itemsize=2, run=1, start=0, window=0,
          engines=True, host="blocks", split=False):
    """window: layers moved, from `start` on (0: every layer).  run: length of
    the runs of consecutive block ids.  engines: the copy-engine path, the
    default of the cache configuration, else the zero-copy kernel.  host:
    "blocks" (one block's layers contiguous) or "layers".  split: K and V in
    separate allocations."""
    c = dict(name=name, kind=kind, **model, blocks=blocks, tokens=tokens, itemsize=itemsize,
             run=run, start=start, window=window or model["layers"], engines=engines, host=host,
             split=split)
    if name is None:
        del c["name"]
    return c


def listed():
    return [
        # One freshly filled block of one layer: the smallest call there is,
        # all launch and link latency.
        _case("save_1blk_1layer", "save", LLAMA8B, 1, start=17, window=1, engines=False),
        # A 256-token prefix of one layer, the reference's layer-wise schedule
        # (one call per layer).
        _case("load_16blk_1layer", "load", LLAMA8B, 16, start=5, window=1, engines=False),
        # The 16 MiB op of the CPU-plumbing configuration, copy-engine mode.
        _case("save_64blk_4layers", "save", SMALL, 64),
        # A 256-token request, every layer (32 MiB): the worker benchmark's op.
        _case("load_16blk", "load", LLAMA8B, 16),
        # An 8-bit cache of a tensor-parallel shard (2 KiB chunks), K and V
        # allocated separately, into a layer-wise host cache.
        _case("save_fp8_shard", "save", LLAMA70B_TP8, 173, itemsize=1, host="layers", split=True,
              engines=False),
        # A long request of the tensor-parallel shard: 4 KiB chunks.
        _case("save_shard_512blk", "save", LLAMA70B_TP8, 512),
        # A 8192-token prefix hit of Llama-3-8B (1 GiB), runs of 8 blocks.
        _case("load_512blk", "load", LLAMA8B, 512, run=8),
        # Layer-wise prefix load of 40 blocks beside prefill (80 MiB), on the
        # zero-copy kernel.
        _case("stream_40blk_kernel", "stream", LLAMA8B, 40, engines=False),
        # Layer-wise load of a 4096-token prefix on the copy engines.
        _case("stream_256blk_engines", "stream", LLAMA8B, 256),
        # Packing 1024 blocks (2 GiB) for a peer: HBM-bound.
        _case("gather_1024blk", "gather", LLAMA8B, 1024),
        # Five MLA blocks of 64 tokens (21 MiB) to a peer: a short request.
        _case("gather_mla_5blk", "gather", MLA, 5, tokens=64),
        # Unpacking an 8-bit shard's blocks (2 KiB chunks, 48 MiB).
        _case("scatter_fp8_shard", "scatter", LLAMA70B_TP8, 151, itemsize=1),
    ]


def draw(rng):
    kind = rng.choice(("save", "load", "stream", "gather", "scatter"))
    model = rng.choice((LLAMA8B, LLAMA8B, LLAMA70B_TP8, MLA, SMALL))
    tokens = rng.choice((4, 16, 16, 32, 64))
    itemsize = rng.choice((2, 2, 1))
    kv = 1 if model["mla"] else 2
    block = model["layers"] * kv * tokens * model["heads"] * model["dim"] * itemsize
    most = (1024 if kind in ("gather", "scatter") else 512) * MIB
    size = math.exp(rng.uniform(math.log(MIB // 4), math.log(most)))
    blocks = max(1, min(int(size / block), most // block, 8192))
    if blocks > 8:
        blocks += rng.randrange(-3, 1)
    start, window, engines, host, split = 0, 0, True, "blocks", False
    if kind in ("save", "load"):
        engines = rng.random() < 0.6
        host = rng.choice(("blocks", "blocks", "layers"))
        split = kv == 2 and rng.random() < 0.2
        if rng.random() < 0.3:
            window = rng.choice((1, 2))
            start = rng.randrange(model["layers"] - window + 1)
    elif kind == "stream":
        engines = rng.random() < 0.5
        host = rng.choice(("blocks", "blocks", "layers"))
    return _case(None, kind, model, blocks, tokens=tokens, itemsize=itemsize,
                 run=rng.choice((1, 1, 8)), start=start, window=window, engines=engines,
                 host=host, split=split)


def _sizes(case):
    kv = 1 if case["mla"] else 2
    chunk = case["tokens"] * case["heads"] * case["dim"] * case["itemsize"]
    # caches hold a quarter more blocks than move, in whole runs
    pool = (case["blocks"] + case["blocks"] // 4 + 24) // case["run"] * case["run"]
    return kv, chunk, pool


def _ids(case, pool, gen):
    """`blocks` distinct ids below `pool`, in runs of `run`, runs in random order."""
    run = case["run"]
    starts = torch.randperm(pool // run, generator=gen)[:-(-case["blocks"] // run)] * run
    return (starts[:, None] + torch.arange(run)).reshape(-1)[:case["blocks"]].contiguous()


def _values(shape, itemsize, gen):
    """A device tensor of `shape` bytes holding normal 16- or 8-bit floats, as int64."""
    n = math.prod(shape) // itemsize
    v = torch.randn(n, dtype=torch.bfloat16, device=DEVICE, generator=gen)
    if itemsize == 1:
        v = v.to(torch.float8_e4m3fn)
    return v.view(torch.uint8).view(torch.int64).view(*shape[:-1], shape[-1] // 8)


_stream = None


def _transfer_stream():
    """The program's one stream for transfers beside compute."""
    global _stream
    if _stream is None:
        _stream = c_ext.transfer_stream()
    return _stream


def prepare(case, seed):
    kv, chunk, pool = _sizes(case)
    layers, window, kind = case["layers"], case["window"], case["kind"]
    ids_gen = torch.Generator().manual_seed(seed)
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    to_device = kind in ("load", "stream", "scatter")

    # device cache [layer][K|V][block][chunk], or [layer] x (K, V); the whole
    # engine's cache is one reservation
    shape = (layers, kv, pool, chunk)
    gpu = torch.empty(layers, kv, pool, chunk // 8, dtype=torch.int64, device=DEVICE)
    for l in range(layers):
        if to_device:
            gpu[l].zero_()
        else:
            gpu[l] = _values(shape[1:], case["itemsize"], gen)
    moved = gpu[case["start"]:case["start"] + window]
    if case["split"]:
        ptrs = [moved[l, k].data_ptr() for l in range(window) for k in range(kv)]
    else:
        ptrs = [moved[l].data_ptr() for l in range(window)]
    state = dict(case=case, gpu=gpu, ptrs=torch.tensor(ptrs, dtype=torch.int64).pin_memory(),
                 gids=_ids(case, pool, ids_gen).pin_memory(),
                 gpu_kv=pool * chunk, gpu_block=chunk, chunk=chunk, kv=kv)

    if kind in ("gather", "scatter"):
        buf = (case["blocks"], layers, kv, chunk)
        state["buffer"] = (_values(buf, case["itemsize"], gen) if to_device else
                           torch.zeros(*buf[:-1], chunk // 8, dtype=torch.int64, device=DEVICE))
        return state

    state["cids"] = _ids(case, pool, ids_gen).pin_memory()
    if case["host"] == "blocks":
        host_shape = (pool, layers, kv, chunk)
        state["cpu_block"], state["cpu_layer"], state["cpu_kv"] = layers * kv * chunk, kv * chunk, chunk
    else:
        host_shape = (layers, kv, pool, chunk)
        state["cpu_layer"], state["cpu_kv"], state["cpu_block"] = kv * pool * chunk, pool * chunk, chunk
    host = pinned_empty(math.prod(host_shape) // 8, torch.int64)
    if to_device:
        host.copy_(_values(host_shape, case["itemsize"], gen).view(-1))
    else:
        host.zero_()
    state["host"] = host
    return state


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "gather":
        c_ext.gather_kv_blocks(state["gids"], state["ptrs"], state["gpu_kv"], state["gpu_block"],
                               state["chunk"], state["buffer"], c["mla"])
        return state["buffer"]
    if kind == "scatter":
        c_ext.scatter_kv_blocks(state["gids"], state["ptrs"], state["gpu_kv"],
                                state["gpu_block"], state["chunk"], state["buffer"], c["mla"])
        return state["gpu"]
    if kind == "stream":
        compute = torch.cuda.current_stream()
        with torch.cuda.stream(_transfer_stream()):
            handle = c_ext.transfer_kv_blocks_layerwise(
                state["gids"], state["ptrs"], state["gpu_kv"], state["gpu_block"], state["cids"],
                state["host"], state["cpu_kv"], state["cpu_layer"], state["cpu_block"],
                state["chunk"], c["start"], 1, is_mla=c["mla"], use_ce_transfer=c["engines"])
        for layer in range(handle.num_groups):
            handle.stream_wait(layer, compute)   # layer's prefill would follow
        handle.release()
        return state["gpu"]
    to_device = kind == "load"
    if c["split"]:
        c_ext.transfer_kv_blocks_kv_ptrs(
            state["gids"], state["ptrs"], state["gpu_block"], state["cids"], state["host"],
            state["cpu_kv"], state["cpu_layer"], state["cpu_block"], state["chunk"], c["start"],
            is_host_to_device=to_device, use_ce_transfer=c["engines"], is_mla=c["mla"])
    else:
        c_ext.transfer_kv_blocks(
            state["gids"], state["ptrs"], state["gpu_kv"], state["gpu_block"], state["cids"],
            state["host"], state["cpu_kv"], state["cpu_layer"], state["cpu_block"],
            state["chunk"], c["start"], is_host_to_device=to_device,
            use_ce_transfer=c["engines"], is_mla=c["mla"])
    return state["gpu"] if to_device else state["host"]


def work(case):
    kv, chunk, _ = _sizes(case)
    # every moved byte is read once and written once
    return {"bytes": 2 * case["blocks"] * case["window"] * kv * chunk, "flops": 0}


def tolerance(case):
    return "exact"
