"""Waiting transfers return when the launch says that everything is there: what the host reads right
behind a put, and what any stream reads right behind a get, is all of it."""
import threading

import numpy as np
import pytest
import torch

from kvsetup import KVSetup, TRTLLM, VLLM, block_ids

pytestmark = pytest.mark.gpu

POLICIES = dict(default={}, confined=dict(arbiter=2), safety_net=dict(arbiter=3), everywhere=dict(arbiter=0),
                claimed=dict(arbiter=0, all_claims_per_wg=8), fat=dict(d2h_wg_threads=256, h2d_wg_threads=256),
                quiet=dict(quiet_wait_us=-100))


@pytest.mark.parametrize("policy", list(POLICIES))
@pytest.mark.parametrize("layers,kv,chunk,n", [(1, 1, 16, 1), (3, 1, 24, 5), (8, 2, 2304, 21),
                                               (4, 2, 8192, 3), (32, 2, 32768, 5), (2, 1, 16400, 600),
                                               (700, 2, 256, 3)])  # more pairs than a launch takes
def test_nothing_is_missing_when_the_call_returns(gpu_device, layers, kv, chunk, n, policy):
    from flexkv_amd.c_ext import launch_policy
    s = KVSetup(VLLM, layers, kv, n + 3, n + 2, chunk, "BLOCKFIRST", seed=n)
    dev = s.to_device(gpu_device)
    rng = np.random.default_rng(chunk)
    elsewhere = torch.cuda.Stream()
    with launch_policy(**POLICIES[policy]):
        for rep in range(4):
            gids, cids = block_ids(rng, n + 3, n), block_ids(rng, n + 2, n)
            dev.host.zero_()
            s.host_ref[:] = 0
            dev.transfer(gids, cids, is_h2d=False)
            put = dev.host_bytes().copy()  # straight away
            s.oracle_transfer(gids, cids, is_h2d=False)
            np.testing.assert_array_equal(put, s.host_ref)
            gids = block_ids(rng, n + 3, n)
            dev.transfer(gids, cids, is_h2d=True)
            with torch.cuda.stream(elsewhere):
                got = [t.cpu().numpy() for t in dev.gpu]
            s.oracle_transfer(gids, cids, is_h2d=True)
            for g, want in zip(got, s.gpu_ref):
                np.testing.assert_array_equal(g, want)


def test_threads_that_wait_at_once(gpu_device):
    """More calls in flight than a set of words holds, on streams of their own, both directions."""
    setups = [KVSetup(TRTLLM, 3, 1, 9, 9, 8192 + 16 * i, "BLOCKFIRST", seed=i) for i in range(70)]
    devs = [s.to_device(gpu_device) for s in setups]
    torch.cuda.synchronize()
    gate, errors = threading.Barrier(len(devs)), []

    def work(i):
        try:
            rng = np.random.default_rng(i)
            with torch.cuda.stream(torch.cuda.Stream()):
                gate.wait()
                for h2d in (False, True, False):
                    gids, cids = block_ids(rng, 9, 5), block_ids(rng, 9, 5)
                    devs[i].transfer(gids, cids, is_h2d=h2d)
                    setups[i].oracle_transfer(gids, cids, is_h2d=h2d)
                    if not h2d:
                        np.testing.assert_array_equal(devs[i].host_bytes(), setups[i].host_ref)
        except BaseException as e:  # noqa: BLE001
            errors.append((i, e))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(devs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors[:2]
    torch.cuda.synchronize()
    for d in devs:
        d.assert_matches_reference()


@pytest.mark.parametrize("policy", ["default", "everywhere", "claimed"])
def test_a_put_larger_than_the_caches_is_all_there(gpu_device, policy):
    """192 MiB, many times what the L2s hold: most lines leave them before the release that the
    word stands behind.  (On three XCDs, on all, and in many small ranges, several launches on one word.)"""
    from flexkv_amd.c_ext import launch_policy
    s = KVSetup(VLLM, 8, 2, 100, 96, 131072, "BLOCKFIRST", seed=96)
    dev = s.to_device(gpu_device)
    rng = np.random.default_rng(96)
    with launch_policy(**POLICIES[policy]):
        for rep in range(3):
            gids, cids = block_ids(rng, 100, 96), block_ids(rng, 96, 96)
            dev.host.fill_(rep)
            dev.transfer(gids, cids, is_h2d=False)
            put = dev.host_bytes().copy()  # straight away
            s.oracle_transfer(gids, cids, is_h2d=False)
            assert np.array_equal(put, s.host_ref)


@pytest.mark.parametrize("policy", ["default", "everywhere", "claimed", "confined", "fat"])
def test_puts_next_to_compute_that_holds_the_compute_units(gpu_device, policy):
    """Workgroups that find no room until others of their launch have ended: each put is all there when
    its call returns, many of them on one word."""
    from flexkv_amd.c_ext import launch_policy
    s = KVSetup(VLLM, 8, 2, 24, 20, 24592, "BLOCKFIRST", seed=24)
    dev = s.to_device(gpu_device)
    rng = np.random.default_rng(24)
    a = torch.randn(4096, 4096, device=gpu_device, dtype=torch.bfloat16)
    out, beside, own = torch.empty_like(a), torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with launch_policy(**POLICIES[policy]):
        for rep in range(12):
            with torch.cuda.stream(beside):
                for _ in range(6):
                    torch.mm(a, a, out=out)
            n = int(rng.integers(1, 20))
            gids, cids = block_ids(rng, 24, n), block_ids(rng, 20, n)
            dev.host.fill_(rep)
            s.host_ref[:] = rep
            with torch.cuda.stream(own):
                dev.transfer(gids, cids, is_h2d=False)
            put = dev.host_bytes().copy()  # straight away
            s.oracle_transfer(gids, cids, is_h2d=False)
            assert np.array_equal(put, s.host_ref), (rep, n)
    torch.cuda.synchronize()
