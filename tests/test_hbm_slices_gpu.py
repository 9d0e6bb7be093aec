"""Engine blocks <-> a dense device buffer at the sizes where the cut into slices can go wrong,
against torch's own indexing: a chunk of exactly a slice, a vector more, a short last slice, one
vector per lane twice as deep, a single slice, and enough bytes for the few-workgroups form."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [  # layers, kv, chunk, blocks
    (1, 1, 8192, 1), (3, 2, 8192, 5), (3, 2, 8208, 5), (5, 1, 18432, 33), (2, 2, 16384, 300),
    (61, 1, 73728, 3), (4, 2, 32768, 257), (3, 2, 8192 + 16 * 511, 7), (2, 1, 32768, 1100),
    (1, 1, 16, 9),  # below a slice: the packed form
]


@pytest.mark.parametrize("unroll", [8, 16])
@pytest.mark.parametrize("to_engine", [False, True])
@pytest.mark.parametrize("layers,kv,chunk,n", SHAPES)
def test_transform_by_slices(gpu_device, layers, kv, chunk, n, to_engine, unroll):
    from flexkv_amd.c_ext import launch_policy, layout_transform
    pool = n + 3
    gen = torch.Generator(device="cuda").manual_seed(chunk + n)
    words = lambda *shape: torch.randint(-2 ** 62, 2 ** 62, shape, device="cuda",  # noqa: E731
                                         generator=gen)
    engine = words(layers, kv, pool, chunk // 8)
    buffer = words(n, layers, kv, chunk // 8)
    ids = torch.randperm(pool, generator=torch.Generator().manual_seed(n))[:n].contiguous()
    want_engine, want_buffer = engine.clone(), buffer.clone()
    on_gpu = ids.to(gpu_device)
    if to_engine:
        want_engine[:, :, on_gpu] = buffer.permute(1, 2, 0, 3)
    else:
        want_buffer = engine[:, :, on_gpu].permute(2, 0, 1, 3).contiguous()
    ptrs = torch.tensor([engine[i].data_ptr() for i in range(layers)], dtype=torch.int64)
    with launch_policy(hbm_unroll=unroll):
        layout_transform(buffer, kv * chunk, chunk, layers * kv * chunk, chunk, ptrs, pool * chunk,
                         chunk, kv * pool * chunk, ids, layers, kv, to_engine, 0)
    torch.cuda.synchronize()
    assert torch.equal(engine, want_engine) and torch.equal(buffer, want_buffer)
