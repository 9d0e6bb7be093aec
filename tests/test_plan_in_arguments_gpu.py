"""Launches whose tables travel in their arguments (up to 400 words: two per (layer, kv) pair, one
per block id) and those whose tables just do not fit any more, against the oracle."""
import numpy as np
import pytest
import torch

from kvsetup import KVSetup, SGLANG, TRTLLM, VLLM, block_ids

pytestmark = pytest.mark.gpu


# engine, layers, kv, chunk, blocks: 2 * layers * kv + 2 * blocks words
SHAPES = [
    (VLLM, 1, 1, 16, 1),            # the smallest there is
    (SGLANG, 50, 2, 2304, 100),     # 400: the last that fits, packed
    (SGLANG, 50, 2, 2304, 101),     # 402: the first that does not
    (VLLM, 199, 1, 8208, 1),        # all pairs, a short last slice
    (TRTLLM, 100, 2, 8192, 1),      # 402, one slice a chunk
    (VLLM, 1, 1, 16384, 199),       # all blocks
    (VLLM, 3, 1, 24, 20),           # vectors of 8 bytes: never in the arguments
]


@pytest.mark.parametrize("sync", [True, False])
@pytest.mark.parametrize("backend,layers,kv,chunk,n", SHAPES)
def test_transfers_around_the_limit(gpu_device, backend, layers, kv, chunk, n, sync):
    s = KVSetup(backend, layers, kv, n + 3, n + 2, chunk, "BLOCKFIRST", seed=layers + n)
    dev = s.to_device(gpu_device)
    rng = np.random.default_rng(n)
    for h2d in (False, True, False, True):  # calls in a row: nothing of one is left for the next
        gids, cids = block_ids(rng, n + 3, n), block_ids(rng, n + 2, n)
        dev.transfer(gids, cids, is_h2d=h2d, sync=sync)
        s.oracle_transfer(gids, cids, is_h2d=h2d)
    torch.cuda.synchronize()
    dev.assert_matches_reference()


@pytest.mark.parametrize("shared", [True, False])
@pytest.mark.parametrize("layers,n", [((30, 31, 30), 64),    # 310 words with shared ids, 566 without
                                      ((30, 31, 30), 109),   # 400 with shared ids
                                      ((30, 31, 30), 110),   # 402
                                      ((2, 1, 3, 2), 1)])
def test_several_jobs_around_the_limit(gpu_device, layers, n, shared):
    from flexkv_amd.c_ext import get_stats, reset_stats, transfer_kv_blocks_multi
    chunks = (18432, 2304, 2048, 8208)
    groups = [KVSetup(VLLM, L, 1, n + 4, n + 4, c, "BLOCKFIRST", seed=L + c)
              for L, c in zip(layers, chunks)]
    devs = [g.to_device(gpu_device) for g in groups]
    rng = np.random.default_rng(n)
    for h2d in (False, True, True):
        ids = [(block_ids(rng, n + 4, n), block_ids(rng, n + 4, n)) for _ in groups]
        if shared:
            ids = [ids[0]] * len(groups)
        calls = [((torch.from_numpy(g), d.ptrs, s.gpu_kv_stride, s.gpu_block_stride,
                   s.gpu_layer_stride, torch.from_numpy(c), d.host, s.cpu_kv_stride,
                   s.cpu_layer_stride, s.cpu_block_stride, s.chunk, 0, s.num_layers),
                  dict(is_host_to_device=h2d, kv_dim=1, gpu_block_type=VLLM, is_blockfirst=True))
                 for s, d, (g, c) in zip(groups, devs, ids)]
        reset_stats()
        transfer_kv_blocks_multi(calls)
        assert get_stats()["kernel_launches"] == 1
        for s, (g, c) in zip(groups, ids):
            s.oracle_transfer(g, c, is_h2d=h2d)
    torch.cuda.synchronize()
    for d in devs:
        d.assert_matches_reference()


@pytest.mark.parametrize("layers,kv,chunk,n", [(1, 1, 16, 1), (64, 2, 8192, 144), (64, 2, 8192, 145),
                                               (3, 1, 18432, 394), (3, 1, 2304, 395)])
def test_transforms_around_the_limit(gpu_device, layers, kv, chunk, n):
    from flexkv_amd.c_ext import layout_transform
    s = KVSetup(VLLM, layers, kv, n + 3, 1, chunk, "BLOCKFIRST", seed=n)
    dev = s.to_device(gpu_device)
    block = layers * kv * chunk
    rng = np.random.default_rng(n)
    buf = torch.zeros(n * block, dtype=torch.uint8, device=gpu_device)
    want = np.stack([a.reshape(kv, n + 3, chunk) for a in s.gpu_ref])  # [layer, kv, block, chunk]
    for to_engine in (False, True, False):
        ids = block_ids(rng, n + 3, n)
        layout_transform(buf, kv * chunk, chunk, block, chunk, dev.ptrs, s.gpu_kv_stride,
                         s.gpu_block_stride, s.gpu_layer_stride, torch.from_numpy(ids), layers, kv,
                         to_engine, VLLM)
        if to_engine:
            want[:, :, ids] = rows.transpose(1, 2, 0, 3)
        else:
            rows = want[:, :, ids].transpose(2, 0, 1, 3).copy()
    np.testing.assert_array_equal(buf.cpu().numpy(), rows.reshape(-1))
    for got, ref in zip(dev.gpu_bytes(), want):
        np.testing.assert_array_equal(got, ref.reshape(-1))


@pytest.mark.parametrize("blocks", [1, 399, 400, 401])
def test_payloads_and_chunk_tables_around_the_limit(gpu_device, blocks):
    from flexkv_amd.c_ext import build_gpu_chunk_ptrs, staging_transfer
    cap, pool = 64, blocks + 2
    rng = np.random.default_rng(blocks)
    ids = torch.from_numpy(block_ids(rng, pool, blocks))
    staging = torch.randint(0, 256, (blocks, cap), dtype=torch.uint8, device=gpu_device)
    sizes = torch.randint(0, cap + 1, (blocks,), device=gpu_device)
    host = torch.zeros((pool, cap), dtype=torch.uint8).pin_memory()
    table = torch.zeros(pool, dtype=torch.int32).pin_memory()
    staging_transfer(staging, cap, sizes, host, cap, None, cap, cap, cap, ids, table, 1, 1, 0, 1, 0,
                     blocks, True, sync=True)
    want = torch.where(torch.arange(cap) < sizes.cpu()[:, None], staging.cpu(), 0)
    assert torch.equal(host[ids], want) and torch.equal(table[ids], sizes.cpu().to(torch.int32))
    back, back_sizes = torch.zeros_like(staging), torch.zeros_like(sizes)
    staging_transfer(back, cap, back_sizes, host, cap, None, cap, cap, cap, ids, table, 1, 1, 0, 1, 0,
                     blocks, False, sync=True)
    assert torch.equal(back.cpu(), want) and torch.equal(back_sizes, sizes)
    out = torch.zeros(2 * blocks, dtype=torch.int64, device=gpu_device)
    ptrs = torch.tensor([1 << 20, 1 << 30], dtype=torch.int64)  # addresses are only computed
    build_gpu_chunk_ptrs(out, ptrs, 0, cap, 0, ids, 0, 1, 0, 2 * blocks, 2, VLLM, sync=True)
    assert torch.equal(out.cpu(), (ptrs[:, None] + ids * cap).flatten())
