"""A layerwise restore that goes out as one launch announcing its batches itself: bytes against
the oracle, the layers a gated consumer sees, the eventfds, batch times, at the sizes where the
cut into batches, ranges and slices can go wrong."""
import os

import numpy as np
import pytest
import torch

from kvsetup import KVSetup, SGLANG, TRTLLM, VLLM

pytestmark = pytest.mark.gpu

# engine, layers, kv, chunk, blocks, layers per batch
SHAPES = [
    (VLLM, 2, 1, 8192, 1, 1),           # a slice a batch: fewer than workgroups
    (VLLM, 5, 2, 8208, 7, 2),           # a vector behind the slice, a short last batch
    (VLLM, 9, 1, 18432, 33, 1),         # 8 + 8 + 2 KiB
    (SGLANG, 4, 2, 73728, 3, 3),
    (TRTLLM, 3, 2, 16384, 129, 1),
    (VLLM, 3, 1, 8192, 1025, 2),        # more blocks than an id tile, above the home-XCD size
    (VLLM, 600, 1, 8192, 2, 7),         # many batches
    (VLLM, 33, 1, 16384, 1, 32),        # a last batch of a single block and layer
    (SGLANG, 11, 2, 18432, 9, 5),
]
POLICIES = dict(default={}, confined=dict(arbiter=2), safety_net=dict(arbiter=3),
                everywhere=dict(arbiter=0))


def restore(grp, s, gids, cids, gran, notify):
    e = torch.empty(0, dtype=torch.int64)
    grp.layerwise_transfer(
        e, e, 0, 0, 0, 0, 0, torch.as_tensor(gids), torch.as_tensor(cids), s.cpu_kv_stride,
        s.cpu_layer_stride, s.cpu_block_stride, s.chunk, s.cpu_kv_stride, s.cpu_layer_stride,
        s.cpu_block_stride, 4, False, s.num_layers, gran, s.kv_dim, 1, counter_id=0,
        kv_shared_across_ranks_mode="sharded", notify_mode=notify)


@pytest.mark.parametrize("policy", list(POLICIES))
@pytest.mark.parametrize("backend,layers,kv,chunk,n,gran", SHAPES)
def test_restore_in_one_launch(gpu_device, backend, layers, kv, chunk, n, gran, policy):
    from flexkv_amd.c_ext import LayerwiseTransferGroup, get_stats, launch_policy, reset_stats
    from flexkv_amd.transfer.eventfd_channel import make_eventfd
    pool = n + 5
    s = KVSetup(backend, layers, kv, pool, pool, chunk, "BLOCKFIRST", seed=chunk + n)
    dev = s.to_device(gpu_device)
    fds = [make_eventfd() for _ in range(layers)]
    i64 = lambda v: torch.tensor([v], dtype=torch.int64)  # noqa: E731
    grp = LayerwiseTransferGroup(
        num_gpus=1, gpu_blocks=[dev.gpu], cpu_blocks=dev.host, ssd_files={}, num_layers=layers,
        gpu_kv_strides_tensor=i64(s.gpu_kv_stride), gpu_block_strides_tensor=i64(s.gpu_block_stride),
        gpu_layer_strides_tensor=i64(s.gpu_layer_stride), gpu_chunk_sizes_tensor=i64(s.chunk),
        iouring_entries=0, iouring_flags=0,
        layer_eventfds_tensor=torch.tensor(fds, dtype=torch.int32), tp_size=1, is_blockfirst=True)
    rng = np.random.default_rng(n)
    consumer = torch.cuda.Stream()
    for rep, notify in enumerate(("polling", "hostfunc", "polling")):
        fresh = rng.integers(0, 256, s.host_bytes, dtype=np.uint8)
        s.host_ref[:] = fresh
        dev.host.copy_(torch.from_numpy(fresh))
        gids = rng.permutation(pool)[:n].astype(np.int64)
        cids = rng.permutation(pool)[:n].astype(np.int64)
        per_layer = backend == VLLM and layers <= 16
        seen = []
        with launch_policy(staged_restore=0, staged_gather=0, **POLICIES[policy]):
            reset_stats()
            torch.cuda.synchronize()
            restore(grp, s, gids, cids, gran, notify)
            with torch.cuda.stream(consumer):
                for l in range(layers):
                    grp.wait_layer(l, consumer)
                    if per_layer:
                        seen.append(dev.gpu[l].clone())
            grp.synchronize()
            consumer.synchronize()
            assert get_stats()["kernel_launches"] == 1
        s.oracle_transfer(gids, cids, True)
        dev.assert_matches_reference(f"restore {rep}")
        for l, t in enumerate(seen):  # what the consumer saw of layer l is all of it
            assert torch.equal(t, dev.gpu[l]), (rep, l)
        for l, fd in enumerate(fds):
            os.set_blocking(fd, False)
            assert int.from_bytes(os.read(fd, 8), "little") == 1, (rep, l)
        times = grp.batch_times_ms()
        assert len(times) == -(-layers // gran) and times[0] >= 0
        assert all(b >= a for a, b in zip(times, times[1:]))
    grp.close()
    for fd in fds:
        os.close(fd)


@pytest.mark.parametrize("layers,blocks", [(24, 16), (61, 3), (40, 64)])
def test_a_consumer_of_one_layer_has_all_before_it(gpu_device, layers, blocks):
    """A stream that waits for one layer only, the last or one in the middle, sees every layer up
    to it: batches of few ranges, many of them under way together."""
    from flexkv_amd.c_ext import LayerwiseTransferGroup, get_stats, launch_policy, reset_stats
    chunk, pool = 16384, blocks + 4
    s = KVSetup(VLLM, layers, 1, pool, pool, chunk, "BLOCKFIRST", seed=layers)
    dev = s.to_device(gpu_device)
    i64 = lambda v: torch.tensor([v], dtype=torch.int64)  # noqa: E731
    grp = LayerwiseTransferGroup(
        num_gpus=1, gpu_blocks=[dev.gpu], cpu_blocks=dev.host, ssd_files={}, num_layers=layers,
        gpu_kv_strides_tensor=i64(s.gpu_kv_stride), gpu_block_strides_tensor=i64(s.gpu_block_stride),
        gpu_layer_strides_tensor=i64(s.gpu_layer_stride), gpu_chunk_sizes_tensor=i64(s.chunk),
        iouring_entries=0, iouring_flags=0, layer_eventfds_tensor=torch.empty(0, dtype=torch.int32),
        tp_size=1, is_blockfirst=True)
    rng = np.random.default_rng(layers)
    consumer = torch.cuda.Stream()
    seen = [torch.empty_like(t) for t in dev.gpu]
    for rep in range(6):
        last = layers - 1 if rep % 2 == 0 else layers // 2
        dev.host.copy_(torch.from_numpy(rng.integers(0, 256, s.host_bytes, dtype=np.uint8)))
        ids = [rng.permutation(pool)[:blocks].astype(np.int64) for _ in range(2)]
        with launch_policy(staged_restore=0, staged_gather=0):
            reset_stats()
            torch.cuda.synchronize()
            restore(grp, s, *ids, 1, "polling")
            with torch.cuda.stream(consumer):
                grp.wait_layer(last, consumer)
                for l in range(last + 1):
                    seen[l].copy_(dev.gpu[l])
            consumer.synchronize()
            grp.synchronize()
            assert get_stats()["kernel_launches"] == 1
        for l in range(last + 1):
            assert torch.equal(seen[l], dev.gpu[l]), (rep, l)
    grp.close()


def vllm_group(s, dev, layers):
    from flexkv_amd.c_ext import LayerwiseTransferGroup
    i64 = lambda v: torch.tensor([v], dtype=torch.int64)  # noqa: E731
    return LayerwiseTransferGroup(
        num_gpus=1, gpu_blocks=[dev.gpu], cpu_blocks=dev.host, ssd_files={}, num_layers=layers,
        gpu_kv_strides_tensor=i64(s.gpu_kv_stride), gpu_block_strides_tensor=i64(s.gpu_block_stride),
        gpu_layer_strides_tensor=i64(s.gpu_layer_stride), gpu_chunk_sizes_tensor=i64(s.chunk),
        iouring_entries=0, iouring_flags=0, layer_eventfds_tensor=torch.empty(0, dtype=torch.int32),
        tp_size=1, is_blockfirst=True)


def test_groups_restoring_at_once(gpu_device):
    """Three groups, a thread and a consumer stream each, at the same time; then the words of the
    groups go to new ones."""
    import threading
    from flexkv_amd.c_ext import launch_policy
    layers, blocks = 12, 24
    failures = []

    def restores(seed):
        try:
            s = KVSetup(VLLM, layers, 1, 32, 32, 16384, "BLOCKFIRST", seed=seed)
            dev = s.to_device(gpu_device)
            consumer, rng = torch.cuda.Stream(), np.random.default_rng(seed)
            for _ in range(2):
                grp = vllm_group(s, dev, layers)
                for rep in range(5):
                    fresh = rng.integers(0, 256, s.host_bytes, dtype=np.uint8)
                    s.host_ref[:] = fresh
                    dev.host.copy_(torch.from_numpy(fresh))
                    ids = [rng.permutation(32)[:blocks].astype(np.int64) for _ in range(2)]
                    restore(grp, s, *ids, 1, "polling" if rep % 2 else "hostfunc")
                    with torch.cuda.stream(consumer):
                        grp.wait_layer(layers - 1, consumer)
                        seen = [t.clone() for t in dev.gpu]
                    consumer.synchronize()
                    grp.synchronize()
                    s.oracle_transfer(*ids, True)
                    dev.assert_matches_reference(f"group {seed} restore {rep}")
                    for l, t in enumerate(seen):
                        assert torch.equal(t, dev.gpu[l]), (seed, rep, l)
                grp.close()
        except BaseException as e:  # noqa: B902 - handed to the test's thread
            failures.append(e)

    with launch_policy(staged_restore=0, staged_gather=0):
        threads = [threading.Thread(target=restores, args=(60 + k,)) for k in range(3)]
        [t.start() for t in threads]
        [t.join() for t in threads]
    if failures:
        raise failures[0]


def test_wait_layer_while_the_stream_is_captured(gpu_device):
    """The wait of a captured stream is the runtime's business, as an event from outside the
    capture is; the graph holds none of the words, and restores before and after are whole."""
    from flexkv_amd.c_ext import launch_policy
    layers, blocks = 9, 7
    s = KVSetup(VLLM, layers, 1, 12, 12, 16384, "BLOCKFIRST", seed=77)
    dev = s.to_device(gpu_device)
    grp = vllm_group(s, dev, layers)
    rng = np.random.default_rng(78)
    stream, counter = torch.cuda.Stream(), torch.zeros(4, device=gpu_device)
    with launch_policy(staged_restore=0, staged_gather=0):
        for rep in range(3):
            fresh = rng.integers(0, 256, s.host_bytes, dtype=np.uint8)
            s.host_ref[:] = fresh
            dev.host.copy_(torch.from_numpy(fresh))
            ids = [rng.permutation(12)[:blocks].astype(np.int64) for _ in range(2)]
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.stream(stream):
                restore(grp, s, *ids, 1, "polling")
                graph.capture_begin(capture_error_mode="thread_local")
                counter.add_(1)
                try:
                    grp.wait_layer(layers - 1, stream)
                except RuntimeError:
                    pass
                graph.capture_end()
                grp.wait_layer(layers - 1, stream)
                seen = [t.clone() for t in dev.gpu]
            grp.synchronize()
            torch.cuda.synchronize()
            s.oracle_transfer(*ids, True)
            dev.assert_matches_reference(f"restore {rep}")
            for l, t in enumerate(seen):
                assert torch.equal(t, dev.gpu[l]), (rep, l)
            before = float(counter[0])
            for k in range(3):
                graph.replay()
                torch.cuda.synchronize()
                assert float(counter[0]) == before + k + 1
    grp.close()


def test_shapes_that_go_batch_by_batch(gpu_device):
    """Few batches of short chunks, and odd vector widths, keep a launch a batch."""
    from flexkv_amd.c_ext import get_stats, launch_policy, reset_stats
    from flexkv_amd.c_ext import LayerwiseTransferGroup
    i64 = lambda v: torch.tensor([v], dtype=torch.int64)  # noqa: E731
    for chunk in (2304, 8200):
        s = KVSetup(VLLM, 3, 1, 9, 9, chunk, "BLOCKFIRST", seed=chunk)
        dev = s.to_device(gpu_device)
        grp = LayerwiseTransferGroup(
            num_gpus=1, gpu_blocks=[dev.gpu], cpu_blocks=dev.host, ssd_files={}, num_layers=3,
            gpu_kv_strides_tensor=i64(s.gpu_kv_stride),
            gpu_block_strides_tensor=i64(s.gpu_block_stride),
            gpu_layer_strides_tensor=i64(s.gpu_layer_stride),
            gpu_chunk_sizes_tensor=i64(s.chunk), iouring_entries=0, iouring_flags=0,
            layer_eventfds_tensor=torch.empty(0, dtype=torch.int32), tp_size=1, is_blockfirst=True)
        ids = np.arange(9, dtype=np.int64)[::-1].copy()
        with launch_policy(staged_restore=0, staged_gather=0):
            reset_stats()
            restore(grp, s, ids, ids, 1, "hostfunc")
            assert get_stats()["kernel_launches"] == 3
        grp.synchronize()
        s.oracle_transfer(ids, ids, True)
        dev.assert_matches_reference(f"chunk {chunk}")
        grp.close()


# chunks of no whole number of slices: pieces that cross chunks, blocks, id tiles and the end of a batch
@pytest.mark.parametrize("policy", ["default", "confined"])
@pytest.mark.parametrize("backend,layers,kv,chunk,n,gran", [
    (VLLM, 4, 1, 16, 1, 1),         # a vector a batch: one short piece, one range
    (VLLM, 4, 1, 2304, 9, 1),       # the fewest batches
    (VLLM, 9, 2, 2304, 57, 2),      # two layers a batch and a short last batch
    (SGLANG, 5, 2, 8176, 3, 1),     # a vector less than a slice
    (TRTLLM, 6, 1, 9936, 21, 1),    # a slice and more
    (VLLM, 5, 1, 48, 3000, 1),      # pieces of 171 blocks: every third id tile starts inside one
    (VLLM, 33, 1, 18432, 40, 1),
    (VLLM, 500, 2, 256, 1, 1),      # more batches than a wavefront has lanes
])
def test_packed_restore_in_one_launch(gpu_device, backend, layers, kv, chunk, n, gran, policy):
    test_restore_in_one_launch(gpu_device, backend, layers, kv, chunk, n, gran, policy)
