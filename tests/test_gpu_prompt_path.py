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
