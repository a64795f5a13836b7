"""The prompt's way through the engine on the GPU: workspace memory, the copy to the host store, the factorisation's
matrix-core kernels at the edges of their tiles."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from lrqk_amd import ops as o
    return o


@pytest.mark.parametrize("streams", [1, 2])
def test_workspace_memory_is_the_caching_allocators(ops, streams):
    """A workspace's blocks come from torch's allocator and go back with it, also after calls on two streams; the
    results do not change when the blocks are handed out again with their old contents."""
    gen = torch.Generator(device=DEV).manual_seed(5)
    scores = torch.randn((2, 3, 5000), generator=gen, device=DEV)
    want = torch.sort(torch.topk(scores, 512, dim=-1).indices, dim=-1).values.to(torch.int32)
    torch.cuda.synchronize()
    for _ in range(3):
        before = torch.cuda.memory_allocated()
        ws = ops.Workspace()
        for i in range(streams):
            with torch.cuda.stream(torch.cuda.Stream() if i else torch.cuda.current_stream()):
                got = ops.select_from_scores(ws, scores, 512)
                torch.cuda.current_stream().synchronize()
            assert torch.equal(got, want)
        held = torch.cuda.memory_allocated()
        assert held > before + got.numel() * 4
        del got
        ws.close()
        assert torch.cuda.memory_allocated() == before


@pytest.mark.parametrize("heads,l,d,dtype", [(3, 1, 16, torch.bfloat16), (2, 257, 80, torch.bfloat16),
                                             (5, 1023, 64, torch.float32), (1, 4099, 256, torch.float32),
                                             (70, 130, 128, torch.bfloat16)])
def test_prompt_rows_to_the_host_store(ops, heads, l, d, dtype):
    """[K|V] rows in device memory and their copy into rows [row0, row0 + l) of the pinned store: bytes as given, the
    rows around them untouched (row counts around the kernel's groups of four, row widths with idle lanes)."""
    gen = torch.Generator(device=DEV).manual_seed(l)
    k = torch.randn((1, heads, l, d), generator=gen, device=DEV).to(dtype)
    v = torch.randn((1, heads, l, d), generator=gen, device=DEV).to(dtype)
    want = torch.cat([k, v], -1)
    rows = ops.interleave_kv(k, v)
    assert torch.equal(rows, want)
    store = torch.full((1, heads, l + 9, 2 * d), -7.0, dtype=dtype, pin_memory=True)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    ops.store_rows(rows, store, 5, side)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.current_stream().synchronize()
    assert torch.equal(store[:, :, 5:5 + l], want.cpu())
    assert (store[:, :, :5] == -7).all() and (store[:, :, 5 + l:] == -7).all()
    with pytest.raises(ValueError):
        ops.store_rows(rows, store, 10, side)
