"""Workloads of the KV-block transfer path, driven through its public operators.

Every case is what a cache worker or a serving engine does per request: it has engine KV
tensors in HBM, a pinned host pool and two lists of block ids in hand, and makes one call
(or, where both directions are busy, a handful of calls from two threads).  All results are
copies of bytes, so every case is compared exactly.

Shapes are those of this repository's benchmark and tests: 16-token blocks of 8 heads x 128
in bf16 (32 KiB per layer and K or V), 64-token pages (128 KiB), fp8 blocks of 5 MiB,
single-latent layers of 16 or 64 tokens (16 and 72 KiB), and layer groups of 18, 2.25 and
2 KiB chunks.
"""
import concurrent.futures
import os

import torch

from flexkv_amd import c_ext

VLLM, TRTLLM, SGLANG = 0, 1, 2
LAYOUTS = {"vllm": VLLM, "trtllm": TRTLLM, "sglang": SGLANG}
GROUP_SHAPES = ((30, 18432), (31, 2304), (30, 2048))  # (layers, bytes of a chunk)
MIB = 1 << 20


def listed():
    return [
        # A decode step's cache hit of one 16-token block: 2 MiB, all latency.
        dict(name="get_one_block", kind="transfer", layout="vllm", layers=32, kv=2, chunk=32768,
             blocks=1, pool=64, host="scattered", h2d=True, engine="kernel"),
        # The blocks a short turn has filled go to the host: 5 blocks, 10 MiB.
        dict(name="put_few_blocks", kind="transfer", layout="vllm", layers=32, kv=2, chunk=32768,
             blocks=5, pool=64, host="scattered", h2d=False, engine="kernel"),
        # A cached prefix of some 580 tokens comes back in 64-token pages: 72 MiB.
        dict(name="get_pages", kind="transfer", layout="sglang", layers=32, kv=2, chunk=131072,
             blocks=9, pool=64, host="run", h2d=True, engine="kernel"),
        # A prompt of 4096 tokens is written out after prefill: 512 MiB.
        dict(name="put_prompt", kind="transfer", layout="vllm", layers=32, kv=2, chunk=32768,
             blocks=256, pool=512, host="scattered", h2d=False, engine="kernel"),
        # fp8 blocks of 5 MiB each through the copy engines, for an engine that keeps its
        # compute units to itself.
        dict(name="put_fp8_copy_engine", kind="transfer", layout="trtllm", layers=80, kv=2,
             chunk=32768, blocks=37, pool=64, host="run", h2d=False, engine="ce"),
        # A model with three layer groups (latent, window and indexer caches): small chunks,
        # one call for all groups of the op.
        dict(name="get_layer_groups", kind="groups", blocks=64, pool=256, h2d=True),
        # Restores layer by layer, single latent per token: a short prefix to an engine in
        # another process (eventfds) ...
        dict(name="restore_short", kind="restore", layers=8, chunk=16384, blocks=16, pool=64,
             host="run", notify="hostfunc"),
        # ... a longer one whose layers the forward stream of this process waits for ...
        dict(name="restore_mid", kind="restore", layers=32, chunk=16384, blocks=64, pool=128,
             host="run", notify="polling"),
        # ... and a long one out of a host pool after some churn.
        dict(name="restore_scattered", kind="restore", layers=61, chunk=73728, blocks=96, pool=128,
             host="scattered", notify="polling"),
        # Puts and gets at the same time, each direction on a thread and stream of its own.
        dict(name="both_ways", kind="both_ways", layers=32, chunk=32768, requests=6, mean=32,
             pool=512),
        # Engine blocks into the dense device buffer a storage write or a codec works on.
        dict(name="fill_buffer", kind="transform", layout="vllm", layers=32, kv=2, chunk=32768,
             blocks=256, pool=512, to_engine=False),
        # Compressed payloads of 50-90 % of their slots into the host pool.
        dict(name="store_payloads", kind="payloads", layers=16, kv=2, capacity=32768, blocks=64,
             write=True),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, evenly over its logarithm."""
    return min(hi, max(lo, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    kind = rng.choice(["transfer"] * 5 + ["groups", "restore", "restore", "both_ways", "transform",
                       "transform", "payloads"])
    if kind in ("transfer", "transform"):
        layout = rng.choice(["vllm", "trtllm", "sglang"])
        kv = rng.choice([1, 2])
        layers = rng.randint(1, 80)
        chunk = rng.choice([2304, 16384, 18432, 32768, 73728, 131072, 16 * rng.randint(64, 4096)])
        engine = "ce" if kind == "transfer" and rng.random() < 0.2 else "kernel"
        most = 64 * MIB if engine == "ce" else 256 * MIB
        blocks = _log(rng, 1, min(2048, max(1, most // (layers * kv * chunk))))
        case = dict(kind=kind, layout=layout, layers=layers, kv=kv, chunk=chunk, blocks=blocks,
                    pool=blocks + rng.randint(1, blocks + 32))
        if kind == "transform":
            return dict(case, to_engine=rng.random() < 0.5)
        return dict(case, host=rng.choice(["run", "scattered"]), h2d=rng.random() < 0.5,
                    engine=engine)
    if kind == "groups":
        blocks = _log(rng, 1, 256)
        return dict(kind=kind, blocks=blocks, pool=2 * blocks + 16, h2d=rng.random() < 0.5)
    if kind == "restore":
        chunk = rng.choice([2304, 8192, 16384, 18432, 73728])
        layers = rng.randint(4, 80)
        blocks = _log(rng, 4, min(512, 256 * MIB // (layers * chunk)))
        return dict(kind=kind, layers=layers, chunk=chunk, blocks=blocks,
                    pool=blocks + rng.randint(1, blocks), host=rng.choice(["run", "scattered"]),
                    notify=rng.choice(["hostfunc", "polling"]))
    if kind == "both_ways":
        requests, mean = rng.randint(2, 6), rng.randint(2, 24)
        return dict(kind=kind, layers=rng.randint(8, 32), chunk=32768, requests=requests, mean=mean,
                    pool=512)
    return dict(kind=kind, layers=rng.randint(1, 24), kv=rng.choice([1, 2]),
                capacity=rng.choice([8192, 18432, 32768]), blocks=_log(rng, 1, 96),
                write=rng.random() < 0.5)


# ---- what a program has in hand before the call --------------------------------
class Engine:
    """KV tensors of one engine layout in one allocation, as int64 words."""

    def __init__(self, layout, layers, kv, pool, chunk, gen, fill):
        words = layers * kv * pool * chunk // 8
        self.words = _random_words(words, gen) if fill else _zero_words(words)
        base, plane = self.words.data_ptr(), pool * chunk
        if layout == "vllm":        # a tensor per layer, [kv, pool, chunk]
            tensors = [base + i * kv * plane for i in range(layers)]
            self.strides = (plane, chunk, kv * plane)
        elif layout == "trtllm":    # one tensor, [pool, layers, kv, chunk]
            tensors = [base]
            self.strides = (chunk, layers * kv * chunk, kv * chunk)
        else:                       # a tensor per (K or V, layer), [pool, chunk]
            tensors = [base + i * plane for i in range(kv * layers)]
            self.strides = (0, chunk, plane)
        # The pointer table the operators take has two halves, K and V; without V the second
        # one is not used.
        if layout == "sglang" and kv == 1:
            tensors = tensors + tensors
        self.ptrs = torch.tensor(tensors, dtype=torch.int64)


def _random_words(n, gen):
    return torch.randint(-(1 << 63), (1 << 63) - 1, (n,), dtype=torch.int64, device="cuda",
                         generator=gen)


def _zero_words(n):
    return torch.zeros(n, dtype=torch.int64, device="cuda")


def _host_words(n, gen=None):
    """A pinned host pool: random words, or zeros."""
    host = torch.empty(n, dtype=torch.int64, pin_memory=True)
    host.copy_(_random_words(n, gen) if gen is not None else _zero_words(n))
    return host


def _ids(pool, n, cpu_gen):
    return torch.randperm(pool, generator=cpu_gen)[:n].to(torch.int64).contiguous()


def _host_ids(case, cpu_gen):
    """(blocks of the host pool, ids): one run of blocks, or blocks scattered over the pool."""
    n = case["blocks"]
    return (n, torch.arange(n, dtype=torch.int64)) if case["host"] == "run" else \
        (case["pool"], _ids(case["pool"], n, cpu_gen))


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    cpu_gen = torch.Generator().manual_seed(seed)
    return _PREPARE[case["kind"]](case, gen, cpu_gen)


class Transfer:
    def __init__(self, case, gen, cpu_gen):
        layers, kv, chunk = case["layers"], case["kv"], case["chunk"]
        self.h2d = case["h2d"]
        self.engine = Engine(case["layout"], layers, kv, case["pool"], chunk, gen, not self.h2d)
        gpu_ids = _ids(case["pool"], case["blocks"], cpu_gen)
        host_blocks, cpu_ids = _host_ids(case, cpu_gen)
        block = layers * kv * chunk
        self.host = _host_words(host_blocks * block // 8, gen if self.h2d else None)
        self.args = (gpu_ids, self.engine.ptrs, *self.engine.strides, cpu_ids, self.host, chunk,
                     kv * chunk, block, chunk, 0, layers)
        self.kw = dict(transfer_num_cta=4, is_host_to_device=self.h2d,
                       use_ce_transfer=case["engine"] == "ce", kv_dim=kv,
                       num_kv_heads=1 if kv == 1 else 8, gpu_block_type=LAYOUTS[case["layout"]],
                       sync=True, ce_path_opt=True, ce_segment_threshold=8, ce_force_path=-1,
                       ce_enable_memcpy2d=True, is_blockfirst=True)

    def run(self):
        c_ext.transfer_kv_blocks(*self.args, **self.kw)
        return self.engine.words if self.h2d else self.host


class Groups:
    """Layer groups that share the blocks of one host pool, each its own part of a block."""

    def __init__(self, case, gen, cpu_gen):
        self.h2d = case["h2d"]
        pool, block = case["pool"], sum(layers * chunk for layers, chunk in GROUP_SHAPES)
        gpu_ids = _ids(pool, case["blocks"], cpu_gen)
        cpu_ids = _ids(pool, case["blocks"], cpu_gen)
        self.engines = [Engine("vllm", layers, 1, pool, chunk, gen, not self.h2d)
                        for layers, chunk in GROUP_SHAPES]
        self.host = _host_words(pool * block // 8, gen if self.h2d else None)
        flat = self.host.view(torch.uint8)
        kw = dict(transfer_num_cta=4, is_host_to_device=self.h2d, use_ce_transfer=False, kv_dim=1,
                  num_kv_heads=1, gpu_block_type=VLLM, sync=True, is_blockfirst=True)
        self.calls, offset = [], 0
        for (layers, chunk), e in zip(GROUP_SHAPES, self.engines):
            self.calls.append(((gpu_ids, e.ptrs, *e.strides, cpu_ids, flat[offset:], chunk, chunk,
                                block, chunk, 0, layers), kw))
            offset += layers * chunk

    def run(self):
        c_ext.transfer_kv_blocks_multi(self.calls)
        return [e.words for e in self.engines] if self.h2d else self.host


class Restore:
    """A layerwise restore: the group lives as long as the engine's tensors do."""

    def __init__(self, case, gen, cpu_gen):
        layers, chunk, pool = case["layers"], case["chunk"], case["pool"]
        self.layers, self.polling = layers, case["notify"] == "polling"
        self.words = _zero_words(layers * pool * chunk // 8)
        tensors = list(self.words.view(layers, pool, chunk // 8).unbind(0))
        gpu_ids = _ids(pool, case["blocks"], cpu_gen)
        host_blocks, cpu_ids = _host_ids(case, cpu_gen)
        self.host = _host_words(host_blocks * layers * chunk // 8, gen)
        one = lambda v: torch.tensor([v], dtype=torch.int64)  # noqa: E731
        self.fds = [os.eventfd(0, os.EFD_SEMAPHORE | os.EFD_NONBLOCK) for _ in range(layers)]
        self.group = c_ext.LayerwiseTransferGroup(
            num_gpus=1, gpu_blocks=[tensors], cpu_blocks=self.host, ssd_files={}, num_layers=layers,
            gpu_kv_strides_tensor=one(pool * chunk), gpu_block_strides_tensor=one(chunk),
            gpu_layer_strides_tensor=one(pool * chunk), gpu_chunk_sizes_tensor=one(chunk),
            iouring_entries=0, iouring_flags=0,
            layer_eventfds_tensor=torch.tensor(self.fds, dtype=torch.int32), tp_size=1,
            ce_enable_memcpy2d=True, is_blockfirst=True)
        if self.polling:
            self.group.set_compute_stream(torch.cuda.current_stream())
        empty = torch.empty(0, dtype=torch.int64)
        self.args = (empty, empty, 0, 0, 0, 0, 32, gpu_ids, cpu_ids, chunk, chunk, layers * chunk,
                     chunk, chunk, chunk, layers * chunk, 4, False, layers, 1, 1, 1)
        self.kw = dict(counter_id=0, notify_mode=case["notify"])

    def run(self):
        self.group.layerwise_transfer(*self.args, **self.kw)
        if self.polling:  # the forward pass of this process starts each layer when it is there
            for layer in range(self.layers):
                self.group.wait_layer(layer)
        return self.words

    def __del__(self, close_fd=os.close):  # bound here: the module may go first
        if hasattr(self, "group"):
            self.group.close()
        for fd in getattr(self, "fds", ()):
            close_fd(fd)


_lanes = None


def _two_lanes():
    """A thread and a stream for each direction, the streams on different hardware queues:
    what a worker that overlaps the directions keeps."""
    global _lanes
    if _lanes is None:
        first, spare = torch.cuda.Stream(), []
        second = torch.cuda.Stream()
        while not c_ext.streams_run_concurrently(first, second) and len(spare) < 8:
            spare.append(second)
            second = torch.cuda.Stream()
        _lanes = [(concurrent.futures.ThreadPoolExecutor(1), s) for s in (first, second)]
    return _lanes


class BothWays:
    """Requests of random sizes, half of them puts and half gets, all on different blocks."""

    def __init__(self, case, gen, cpu_gen):
        layers, chunk, pool = case["layers"], case["chunk"], case["pool"]
        sizes = torch.empty(2 * case["requests"]).geometric_(1.0 / case["mean"], generator=cpu_gen)
        sizes = sizes.clamp(1, 2 * case["mean"]).to(torch.int64)
        # every seed moves the same number of blocks
        want, n = 2 * case["requests"] * case["mean"], sizes.numel()
        sizes += (want - int(sizes.sum())) // n
        sizes[0] += want - int(sizes.sum())
        sizes.clamp_(min=1)
        self.gets = Engine("vllm", layers, 2, pool, chunk, gen, True)
        block = layers * 2 * chunk
        self.host = _host_words(pool * block // 8, gen)
        gpu_ids, cpu_ids = _ids(pool, pool, cpu_gen), _ids(pool, pool, cpu_gen)
        self.calls, at = ([], []), 0
        for i, size in enumerate(sizes.tolist()):
            kw = dict(transfer_num_cta=4, is_host_to_device=i % 2 == 1, kv_dim=2, num_kv_heads=8,
                      gpu_block_type=VLLM, sync=True, is_blockfirst=True)
            self.calls[i % 2].append(((gpu_ids[at:at + size], self.gets.ptrs, *self.gets.strides,
                                       cpu_ids[at:at + size], self.host, chunk, 2 * chunk, block,
                                       chunk, 0, layers), kw))
            at += size

    @staticmethod
    def _direction(stream, calls):
        with torch.cuda.stream(stream):
            for args, kw in calls:
                c_ext.transfer_kv_blocks(*args, **kw)

    def run(self):
        for job in [pool.submit(self._direction, stream, calls)
                    for (pool, stream), calls in zip(_two_lanes(), self.calls)]:
            job.result()
        return self.gets.words, self.host


class Transform:
    def __init__(self, case, gen, cpu_gen):
        layers, kv, chunk = case["layers"], case["kv"], case["chunk"]
        self.to_engine = case["to_engine"]
        self.engine = Engine(case["layout"], layers, kv, case["pool"], chunk, gen,
                             not self.to_engine)
        block = layers * kv * chunk
        words = case["blocks"] * block // 8
        self.buffer = _random_words(words, gen) if self.to_engine else _zero_words(words)
        self.args = (self.buffer, kv * chunk, chunk, block, chunk, self.engine.ptrs,
                     *self.engine.strides, _ids(case["pool"], case["blocks"], cpu_gen), layers, kv,
                     self.to_engine, LAYOUTS[case["layout"]])

    def run(self):
        c_ext.layout_transform(*self.args)
        return self.engine.words if self.to_engine else self.buffer


class Payloads:
    def __init__(self, case, gen, cpu_gen):
        layers, kv, blocks, cap = case["layers"], case["kv"], case["blocks"], case["capacity"]
        total, pool = layers * kv * blocks, blocks + 8
        self.write = case["write"]
        sizes = torch.randint(cap // 2, cap * 9 // 10, (total,), generator=cpu_gen)
        ids = _ids(pool, blocks, cpu_gen)
        table = torch.zeros((pool, layers, kv), dtype=torch.int32)
        self.staging = _random_words(total * cap // 8, gen) if self.write else \
            _zero_words(total * cap // 8)
        self.host = _host_words(pool * layers * kv * cap // 8, None if self.write else gen)
        if not self.write:  # payload (layer, kv, position) has its size in the table of its block
            table[ids] = sizes.view(layers, kv, blocks).permute(2, 0, 1).to(torch.int32)
        self.table = table.view(-1).pin_memory()
        self.sizes = sizes.cuda() if self.write else torch.zeros(total, dtype=torch.int64,
                                                                 device="cuda")
        self.overflow = torch.zeros(1, dtype=torch.int32, device="cuda")
        self.args = (self.staging, cap, self.sizes, self.host, cap, self.overflow, cap, kv * cap,
                     layers * kv * cap, ids, self.table, layers * kv, kv, 0, kv, 0, total,
                     self.write)

    def run(self):
        c_ext.staging_transfer(*self.args, transfer_num_cta=4)
        return (self.host, self.table) if self.write else (self.staging, self.sizes)


_PREPARE = {"transfer": Transfer, "groups": Groups, "restore": Restore, "both_ways": BothWays,
            "transform": Transform, "payloads": Payloads}


def run(state):
    return state.run()


def work(case):
    """Every byte is read once at one end and written once at the other."""
    kind = case["kind"]
    if kind == "groups":
        moved = case["blocks"] * sum(layers * chunk for layers, chunk in GROUP_SHAPES)
    elif kind == "restore":
        moved = case["blocks"] * case["layers"] * case["chunk"]
    elif kind == "both_ways":
        moved = 2 * case["requests"] * case["mean"] * case["layers"] * 2 * case["chunk"]
    elif kind == "payloads":  # sizes are even between 50 and 90 % of the capacity
        moved = 0.7 * case["blocks"] * case["layers"] * case["kv"] * case["capacity"]
    else:
        moved = case["blocks"] * case["layers"] * case["kv"] * case["chunk"]
    return {"bytes": 2 * moved, "flops": 0}


def tolerance(case):
    return "exact"
