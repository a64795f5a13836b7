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


def test_a_reserved_workspace_goes_without_waiting(ops):
    """Memory that is reserved while a stream is current is that stream's: the workspace is used there and dropped
    without waiting for the device."""
    scores = torch.randn((2, 3, 5000), device=DEV)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        ws = ops.Workspace()
        ws.reserve(6, 5000, 512, 528, 16, 64)
        ops.select_from_scores(ws, scores, 512)
        torch.cuda._sleep(400_000_000)
        busy = torch.cuda.Event()
        busy.record()
        ws.close()
        waited = busy.query()
    torch.cuda.synchronize()
    assert not waited


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


@pytest.mark.parametrize("context,name", [(1000, "kernel"), (9000, "copy engine")])
def test_a_dropped_caches_store_waits_for_its_copies(ops, context, name):
    """A cache that goes while its prompt is still on the way to the host store (written by a kernel or by a copy
    engine): its pinned block is nobody else's before that work is done."""
    from lrqk_amd import DynamicLRQKCache
    gen = torch.Generator(device=DEV).manual_seed(context)
    q = torch.randn((1, 4, context, 64), generator=gen, device=DEV).to(torch.bfloat16)
    k, v = (torch.randn((1, 2, context, 64), generator=gen, device=DEV).to(torch.bfloat16) for _ in range(2))
    for attempt in range(2):   # (the first loads kernels, which waits for the device)
        cache = DynamicLRQKCache(r=16, num_active_tokens=128, max_iter=1, lite_tokens=16, tol=0.0,
                                 max_sequence_length=context + 64, num_key_value_groups=2)
        torch.cuda.synchronize()
        torch.cuda._sleep(400_000_000)   # some tenths of a second
        cache.update(q, k, v, 0)
        store = cache.lwattn[0].KVcpu.data
        place, shape = store.data_ptr(), store.shape
        busy = torch.cuda.Event()
        busy.record()
        del cache, store
        other = torch.empty(shape, dtype=torch.bfloat16, pin_memory=True)
        early = not busy.query()
        same = other.data_ptr() == place
        torch.cuda.synchronize()
        del other
    print(name, "still under way:", early, flush=True)
    assert early and not same


@pytest.mark.parametrize("capacity,tokens", [(9000, 0), (200, 80)])
def test_a_short_prompts_store_waits_for_its_flushes(ops, capacity, tokens):
    """The same for a prompt that fits the active set, whose store only the decode steps' kernels write (a flush of the
    ring per 16 tokens): as it was allocated, and after it has grown (from 200 rows, within 80 tokens)."""
    from lrqk_amd import DynamicLRQKCache
    gen = torch.Generator(device=DEV).manual_seed(capacity)

    def rows(heads, n):
        return torch.randn((1, heads, n, 64), generator=gen, device=DEV).to(torch.bfloat16)
    prompt = rows(4, 140), rows(2, 140), rows(2, 140)
    token = rows(4, 1), rows(2, 1), rows(2, 1)
    for attempt in range(2):   # (the first loads kernels, which waits for the device)
        cache = DynamicLRQKCache(r=16, num_active_tokens=128, max_iter=1, lite_tokens=16, tol=0.0,
                                 max_sequence_length=capacity, num_key_value_groups=2)
        cache.update(*prompt, 0)
        first = cache.lwattn[0].KVcpu.data.data_ptr()
        for _ in range(tokens):
            cache.update(*token, 0)
        torch.cuda.synchronize()
        torch.cuda._sleep(400_000_000)   # some tenths of a second
        for _ in range(20):
            cache.update(*token, 0)
        store = cache.lwattn[0].KVcpu.data
        place, shape = store.data_ptr(), store.shape
        assert (place != first) == (tokens > 0)
        busy = torch.cuda.Event()
        busy.record()
        del cache, store
        other = torch.empty(shape, dtype=torch.bfloat16, pin_memory=True)
        early = not busy.query()
        same = other.data_ptr() == place
        torch.cuda.synchronize()
        del other
    assert early and not same


def test_a_host_ahead_of_the_gpu_holds_few_stores(ops, monkeypatch):
    """A cache per prompt, each dropped before the GPU has come to it: the host waits instead of taking a pinned block for
    every prompt that it is ahead (the newest and one before it here, and one on its way back)."""
    from lrqk_amd import DynamicLRQKCache, buffers
    monkeypatch.setattr(buffers, "_AHEAD_BYTES", 1)
    gen = torch.Generator(device=DEV).manual_seed(1)
    q = torch.randn((1, 4, 3000, 64), generator=gen, device=DEV).to(torch.bfloat16)
    k, v = (torch.randn((1, 2, 3000, 64), generator=gen, device=DEV).to(torch.bfloat16) for _ in range(2))
    places = set()
    for _ in range(8):
        cache = DynamicLRQKCache(r=16, num_active_tokens=128, max_iter=1, lite_tokens=16, tol=0.0,
                                 max_sequence_length=3264, num_key_value_groups=2)
        cache.update(q, k, v, 0)
        places.add(cache.lwattn[0].KVcpu.data.data_ptr())
        torch.cuda._sleep(30_000_000)
        del cache
    torch.cuda.synchronize()
    print("blocks", len(places), flush=True)
    assert len(places) <= 4


def test_stores_of_live_caches_are_not_waited_for(ops, monkeypatch):
    """The host waits for stores that come back, not for those of caches in use: the layers of a model."""
    from lrqk_amd import DynamicLRQKCache, buffers
    monkeypatch.setattr(buffers, "_AHEAD_BYTES", 1)
    gen = torch.Generator(device=DEV).manual_seed(1)
    q = torch.randn((1, 4, 3000, 64), generator=gen, device=DEV).to(torch.bfloat16)
    k, v = (torch.randn((1, 2, 3000, 64), generator=gen, device=DEV).to(torch.bfloat16) for _ in range(2))

    def model():
        return DynamicLRQKCache(r=16, num_active_tokens=128, max_iter=1, lite_tokens=16, tol=0.0, max_sequence_length=3264,
                                num_key_value_groups=2)
    for attempt in range(2):   # (the first loads kernels and takes pinned memory, which waits for the device)
        cache = model()
        torch.cuda.synchronize()
        torch.cuda._sleep(400_000_000)
        slept = torch.cuda.Event()
        slept.record()
        for layer in range(5):
            cache.update(q, k, v, layer)
        waited = slept.query()
        torch.cuda.synchronize()
    assert not waited


@pytest.mark.parametrize("dtype,d,r,l,hq,hkv,iters", [
    (torch.float32, 64, 1, 128, 2, 2, 1),        # the fewest rows the Gram matrices take, one column of factors
    (torch.float32, 64, 16, 129, 6, 2, 2),       # a row beyond whole groups; three query heads per kv head
    (torch.float32, 128, 17, 1000, 4, 4, 2),     # the first rank that is padded to two tiles
    (torch.bfloat16, 64, 32, 4097, 4, 1, 3),     # more than one split
    (torch.bfloat16, 64, 33, 515, 2, 1, 2),      # the first rank that is padded to four tiles
    (torch.bfloat16, 128, 48, 257, 8, 2, 3),
    (torch.float32, 128, 64, 2531, 2, 1, 4),
    (torch.bfloat16, 128, 64, 9001, 2, 1, 4),
    (torch.bfloat16, 128, 24, 1055, 8, 2, 2),    # four and two query heads from one reading of K: rows of whole groups
    (torch.bfloat16, 128, 18, 300, 4, 2, 2),     # of four factors, rows that are none
    (torch.float32, 128, 40, 700, 2, 1, 0),      # no iteration: the given factors are the result
])
def test_fit_on_gram_matrices(ops, oracle, dtype, d, r, l, hq, hkv, iters):
    """Every instance of the streaming kernels and of the fp64 iteration (row widths 64 and 128, ranks padded to 16, 32
    and 64, fp32 and bf16 rows) against the oracle in fp64.  Limit: a sum of up to 1024 rows per wave adds 32 group sums
    in fp32, each group exact to 2^-24 times its terms, so the sums are off by at most 34 x 2^-24 = 2e-6 of their
    terms; random rows of rank above r keep the systems within a factor of ten of that."""
    from lrqk_amd import synth
    gen = torch.Generator().manual_seed(l + r)
    Q, _ = synth.low_rank_noise(gen, 1, hq, l, d, min(d, 2 * r), 0.05, dtype)
    K, _ = synth.low_rank_noise(gen, 1, hkv, l, d, min(d, 2 * r), 0.05, dtype)
    A0 = torch.randn((1, hq, l, r), generator=gen)
    A1 = torch.randn((1, hq, l, r), generator=gen)
    ws = ops.Workspace()
    got = ops.als_prefill(ws, Q.to(DEV), K.to(DEV), A0.to(DEV), A1.to(DEV), iters, 0.0)
    ref = oracle.als_prefill_w1(Q.double(), oracle.repeat_kv(K, hq // hkv).double(), A0.double(), A1.double(), iters, 0.0)
    for name, g, w in zip(("A_Q", "B_Q", "A_K", "B_K"), got, ref):
        off = float((g.cpu().double() - w).norm() / w.norm())
        print(f"{name}: {off:.2e}", flush=True)
        assert off < 2e-5, name
    # the same fit into a cache's buffers: the same numbers in the rows' type, nothing beside them touched
    buf = torch.full((1, hq, l + 7, r), 9.0, dtype=dtype, device=DEV)
    a_q, b_q, a_k, b_k = ops.als_prefill_store(ws, Q.to(DEV), K.to(DEV), A0.to(DEV), A1.to(DEV), iters, 0.0, a_k=buf, row0=3,
                                               last_query_row=True)
    assert torch.equal(a_q, got[0][:, :, -1:].to(dtype)) and torch.equal(buf[:, :, 3:3 + l], got[2].to(dtype))
    assert torch.equal(b_q, got[1].to(dtype)) and torch.equal(b_k, got[3].to(dtype))
    assert (buf[:, :, :3] == 9).all() and (buf[:, :, 3 + l:] == 9).all()


@pytest.mark.parametrize("d,r,heads,tol", [(64, 17, 160, 0.0), (64, 32, 161, 0.0), (128, 32, 96, 0.0), (128, 24, 97, 0.0),
                                           (128, 33, 64, 0.0), (128, 64, 65, 0.0), (64, 64, 1, 0.0), (128, 32, 9, 1e30),
                                           (64, 17, 112, 0.0), (64, 32, 113, 0.0), (64, 33, 80, 0.0), (64, 40, 81, 0.0),
                                           (128, 32, 64, 0.0), (128, 24, 65, 0.0)])
def test_fit_in_slices_and_whole(ops, oracle, d, r, heads, tol):
    """The iteration in slices of a head's columns (up to 64 heads of 128; of 64 up to 112 at ranks to 32, 80 above; head
    counts that are no multiple of the XCDs) and whole (one head more), and a fit that stops at its second iteration:
    against the oracle in fp64, with the limit of the test above."""
    gen = torch.Generator().manual_seed(heads + r)
    from lrqk_amd import synth
    l = 2 * d + 5
    Q, _ = synth.low_rank_noise(gen, 1, heads, l, d, min(d, 2 * r), 0.05, torch.bfloat16)
    K, _ = synth.low_rank_noise(gen, 1, heads, l, d, min(d, 2 * r), 0.05, torch.bfloat16)
    A0, A1 = (torch.randn((1, heads, l, r), generator=gen) for _ in range(2))
    got = ops.als_prefill(ops.Workspace(), Q.to(DEV), K.to(DEV), A0.to(DEV), A1.to(DEV), 3, tol)
    ref = oracle.als_prefill_w1(*(t.to(DEV).double() for t in (Q, K, A0, A1)), 3, tol)
    for name, g, w in zip(("A_Q", "B_Q", "A_K", "B_K"), got, ref):
        off = float(((g.double() - w).flatten(2).norm(dim=2) / w.flatten(2).norm(dim=2)).max())
        print(f"{name}: {off:.2e}", flush=True)
        assert off < 2e-5, name


@pytest.mark.parametrize("d", [64, 128])
def test_sums_over_millions_of_rows(ops, d):
    """However long the prompt, a split adds 4096 rows up in fp32: the given factors of 8M equal rows, whose sums never
    cancel, and the B that follows from them.  Limit: a wave adds 32 groups of 32 rows (d 64: as many; the K side at
    d 128: 16) to its total, each addition off by at most 2^-25 of the total so far, 16 x 2^-24 of it in the end; 8 waves'
    totals, the group's own 32 x 3 products and the last rounding are below 8 x 2^-24; both for A^T A and A^T X."""
    l = 1 << 23
    X = torch.ones((1, 1, l, d), device=DEV, dtype=torch.bfloat16)
    ws = ops.Workspace()
    for a in (1.3, 1.4142135, 1.61803398, 1.9):
        A0 = torch.full((1, 1, l, 1), a, device=DEV)
        got = ops.als_prefill(ws, X, X, A0.clone(), A0.clone(), 0, 0.0)
        for name, g in (("B_Q", got[1]), ("B_K", got[3])):
            off = float((g.double() * float(A0[0, 0, 0, 0]) - 1).abs().max()) * 2 ** 24
            print(f"{name} {a}: {off:.1f} x 2^-24", flush=True)
            assert off < 2 * (16 + 8), name


@pytest.mark.parametrize("d,r", [(64, 16), (128, 48), (32, 8)])
def test_fp32_factors_are_not_copied(ops, monkeypatch, d, r):
    """fp32 results of cast_lrqk_prefill lie where the initial factors lay, and are those of the form that writes them
    into a cache's buffers."""
    from lrqk_amd import cast_lrqk_prefill, factor
    gen = torch.Generator(device=DEV).manual_seed(d)
    Q = torch.randn((1, 4, 300, d), generator=gen, device=DEV)
    K = torch.randn((1, 2, 300, d), generator=gen, device=DEV)
    start = tuple(torch.randn((1, 4, 300, r), generator=gen, device=DEV) for _ in range(2))
    seen, make = [], factor._initial_factors
    monkeypatch.setattr(factor, "_initial_factors", lambda *a: seen.append(make(*a)) or seen[-1])
    got = tuple(cast_lrqk_prefill(Q, K, r, max_iter=2, tol=0.0, init_factors=start))
    want = ops.als_prefill_store(ops.Workspace(), Q, K, start[0].clone(), start[1].clone(), 2, 0.0)
    assert all(torch.equal(g, w) for g, w in zip(got, want))
    assert (got[0].data_ptr(), got[2].data_ptr()) == tuple(t.data_ptr() for t in seen[0])


@pytest.mark.parametrize("d,r,l", [(64, 16, 700), (64, 48, 129), (128, 32, 5000), (128, 64, 2531)])
def test_fp32_rows_are_factorised_row_by_row(ops, monkeypatch, d, r, l):
    """fp32 prompts take the row-by-row formulation, to the bit, at every width and rank that bf16 rows take to Gram
    matrices: an fp32 generation goes on from these factors, and those of the other formulation are 1e-5 away."""
    gen = torch.Generator(device=DEV).manual_seed(d + l)
    Q = torch.randn((1, 4, l, d), generator=gen, device=DEV)
    K = torch.randn((1, 2, l, d), generator=gen, device=DEV)
    A0, A1 = (torch.randn((1, 4, l, r), generator=gen, device=DEV) for _ in range(2))
    ws = ops.Workspace()
    got = ops.als_prefill(ws, Q, K, A0.clone(), A1.clone(), 2, 0.0)
    monkeypatch.setenv("LRQK_PREFILL_ROWWISE", "1")
    want = ops.als_prefill(ws, Q, K, A0.clone(), A1.clone(), 2, 0.0)
    for name, g, w in zip(("A_Q", "B_Q", "A_K", "B_K"), got, want):
        assert torch.equal(g, w), name


@pytest.mark.parametrize("d,r,hq,hkv,l,iters,tol", [
    (128, 64, 4, 2, 33, 2, 0.0), (128, 33, 3, 1, 1000, 2, 0.0), (128, 48, 2, 2, 1, 1, 0.0),    # one row beyond a tile; one row
    (64, 64, 2, 1, 5, 1, 0.0), (64, 40, 4, 1, 257, 0, 0.0), (128, 63, 1, 1, 40000, 1, 0.0),    # 20 partial sums: added in fp64
    (128, 33, 3, 1, 65, 2, 0.0), (64, 64, 3, 3, 97, 2, 0.0),                                   # one row beyond whole tiles, rows enough
    (128, 56, 4, 4, 300, 4, 1e30)])                                                            # stops at its second iteration
def test_wide_fp32_rows_as_the_general_kernel(ops, monkeypatch, d, r, hq, hkv, l, iters, tol):
    """Ranks 33 to 64 of fp32 rows on the matrix cores: the factors of the general kernels, to the bit, also where the rows
    are fewer than the rank and the systems singular; and those of rows that are not 16-byte aligned, which take the general
    pass and the r x r stages of the others."""
    gen = torch.Generator(device=DEV).manual_seed(r + l)
    Q, K = (torch.randn((1, h, l, d), generator=gen, device=DEV) for h in (hq, hkv))
    A0, A1 = (torch.randn((1, hq, l, r), generator=gen, device=DEV) for _ in range(2))

    def off(t):   # the same values 4 bytes beyond a multiple of 16
        return torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)
    ws = ops.Workspace()
    got = ops.als_prefill(ws, Q, K, A0.clone(), A1.clone(), iters, tol)
    unaligned = ops.als_prefill(ws, off(Q), off(K), A0.clone(), A1.clone(), iters, tol)
    monkeypatch.setenv("LRQK_PREFILL_ROWWISE", "general")
    general = ops.als_prefill(ws, Q, K, A0.clone(), A1.clone(), iters, tol)

    def bits(t):   # (a NaN of any payload is a NaN)
        return torch.where(t.isnan(), torch.full_like(t, float("nan")), t).view(torch.int32)
    for name, g, u, w in zip(("A_Q", "B_Q", "A_K", "B_K"), got, unaligned, general):
        print(name, float((~torch.isfinite(g)).float().mean()), flush=True)
        assert torch.isfinite(g).all() or l < r, name
        assert torch.equal(bits(g), bits(w)), name
        assert torch.equal(bits(u), bits(w)), name


@pytest.mark.parametrize("d,r,hq,hkv,l,iters,tol", [
    (128, 16, 6, 2, 1000, 2, 0.0), (128, 1, 2, 1, 33, 1, 0.0), (128, 15, 1, 1, 40000, 1, 0.0),  # 20 partial sums: in fp64
    (64, 16, 4, 4, 257, 3, 0.0), (64, 9, 3, 1, 31, 2, 0.0), (64, 16, 2, 1, 2531, 0, 0.0), (128, 16, 4, 2, 300, 4, 1e30)])
def test_narrow_fp32_rows_as_wide_tiles(ops, d, r, hq, hkv, l, iters, tol):
    """Ranks up to 16 of fp32 rows of 64 and 128 on 16-wide tiles: rows whose last four elements are zero have the factors
    of the 32-wide tiles that rows without them take, to the bit (a product with zero changes no sum)."""
    gen = torch.Generator(device=DEV).manual_seed(r + l)
    Q, K = (torch.randn((1, h, l, d), generator=gen, device=DEV) for h in (hq, hkv))
    Q[..., -4:], K[..., -4:] = 0, 0
    A0, A1 = (torch.randn((1, hq, l, r), generator=gen, device=DEV) for _ in range(2))
    ws = ops.Workspace()
    got = ops.als_prefill(ws, Q, K, A0.clone(), A1.clone(), iters, tol)
    want = ops.als_prefill(ws, Q[..., :-4].contiguous(), K[..., :-4].contiguous(), A0.clone(), A1.clone(), iters, tol)
    for name, g, w in zip(("A_Q", "B_Q", "A_K", "B_K"), got, want):
        if name in ("B_Q", "B_K"):
            assert (g[..., -4:] == 0).all(), name
            g = g[..., :-4]
        assert torch.isfinite(g).all() and torch.equal(g, w), name


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("r,m", [(16, 1025), (16, 4127), (32, 1056), (32, 9001), (64, 1060), (64, 5000)])
def test_selection_through_a_freshly_built_index(ops, dtype, r, m):
    """The index of many rows at once (whole and partial groups of 32, every rank that has one): the selections are
    those of the plain scan, also with rows that are zero, huge, infinite or not numbers, and the bounds are tight
    enough that most rows are never looked at again."""
    gen = torch.Generator(device=DEV).manual_seed(m + r)
    mix = torch.randn((r, r), generator=gen, device=DEV)
    a_k = (torch.randn((1, 3, m + 5, r), generator=gen, device=DEV) @ mix).to(dtype)
    a_k[:, 0, 7] = 0
    a_k[:, 1, 40] *= 3e4
    a_k[:, 2, 33, 1] = float("inf")
    a_k[:, 2, 64, 0] = float("nan")
    q0 = torch.randn((1, 3, 1, r), generator=gen, device=DEV)
    plain, indexed = ops.Workspace(), ops.Workspace()
    indexed.score_index(True)
    for step in range(3):   # (the first scan has no bound yet: every row is a candidate)
        q = (q0 + 0.05 * step).to(dtype)
        want = ops.score_select(plain, a_k, q, m, 100)
        got = ops.score_select(indexed, a_k, q, m, 100)
        assert torch.equal(got, want), step
    rows, rescored = indexed.scan_stats()
    print(f"rescored {rescored} of {rows}", flush=True)
    assert rows == 3 * m and rescored < rows // 3


@pytest.mark.parametrize("dtype,r,heads,m", [
    (torch.bfloat16, 32, 13, 32767), (torch.bfloat16, 32, 13, 32768), (torch.float32, 16, 32, 13311), (torch.float32, 16, 32, 13313),
    (torch.bfloat16, 64, 32, 14001), (torch.bfloat16, 32, 33, 13000), (torch.float32, 32, 1, 425984)])
def test_selection_on_either_side_of_the_scans_orders(ops, dtype, r, heads, m):
    """Scans of 416K rows of up to 32 heads take the heads in a row, others a head after the other: the selections are those
    of the plain scan."""
    gen = torch.Generator(device=DEV).manual_seed(heads + m)
    a_k = torch.randn((1, heads, m + 3, r), generator=gen, device=DEV).to(dtype)
    q0 = torch.randn((1, heads, 1, r), generator=gen, device=DEV)
    plain, indexed = ops.Workspace(), ops.Workspace()
    indexed.score_index(True)
    for step in range(2):
        q = (q0 + 0.05 * step).to(dtype)
        assert torch.equal(ops.score_select(indexed, a_k, q, m, 300), ops.score_select(plain, a_k, q, m, 300)), step
    assert indexed.scan_stats()[0] == heads * m


@pytest.mark.parametrize("dtype,hq,hkv,d,l,k,lite", [(torch.float32, 2, 1, 8, 12, 8, 4), (torch.bfloat16, 6, 2, 64, 515, 33, 7),
                                                     (torch.float32, 4, 4, 256, 300, 100, 1), (torch.bfloat16, 4, 2, 64, 90, 16, 0)])
def test_active_set_of_a_prompt(ops, dtype, hq, hkv, d, l, k, lite):
    """Selected rows, then the last tokens' rows and ids (a prompt that just fills the set, slots beyond whole rounds of
    a workgroup, rows of two and of 128 chunks, no ring)."""
    gen = torch.Generator(device=DEV).manual_seed(l)
    K = torch.randn((2, hkv, l, d), generator=gen, device=DEV).to(dtype)
    V = torch.randn((2, hkv, l, d), generator=gen, device=DEV).to(dtype)
    hit = torch.rand((2, hq, l - lite), generator=gen, device=DEV).argsort(-1)[:, :, :k].sort(-1).values.to(torch.int32)
    ids = torch.cat([hit, torch.arange(l - lite, l, dtype=torch.int32, device=DEV).expand(2, hq, lite)], -1)
    idx = torch.cat([hit, torch.full((2, hq, lite), -1, dtype=torch.int32, device=DEV)], -1).contiguous()
    Ka = torch.empty((2, hq, k + lite, d), dtype=dtype, device=DEV)
    Va = torch.empty_like(Ka)
    ops.fill_active(K, V, idx, Ka, Va, k)
    rows = ids.long().unsqueeze(-1).expand(-1, -1, -1, d)
    g = hq // hkv
    assert torch.equal(idx, ids)
    assert torch.equal(Ka, torch.gather(K.repeat_interleave(g, 1), 2, rows))
    assert torch.equal(Va, torch.gather(V.repeat_interleave(g, 1), 2, rows))


@pytest.mark.parametrize("dtype,batch,hq,hkv,d,l,k,rows", [
    (torch.bfloat16, 1, 4, 2, 64, 1500, 100, 128), (torch.float32, 2, 6, 3, 128, 901, 64, 7), (torch.float32, 1, 2, 2, 8, 700, 33, 1),
    (torch.bfloat16, 3, 8, 2, 64, 1203, 128, 512), (torch.float32, 2, 6, 3, 128, 901, 64, 256),  # heads of several sequences
    (torch.float32, 1, 4, 1, 256, 600, 64, 96),     # (rows wider than the cache takes: it stays empty)
    (torch.bfloat16, 1, 4, 4, 128, 80, 64, 96)])    # (fewer tokens left over than the cache has rows)
def test_cache_filled_by_the_prompt_is_invisible(ops, dtype, batch, hq, hkv, d, l, k, rows):
    """The next best tokens of a prompt in the victim cache change where a missed row comes from and nothing else; and rows
    do come from it."""
    from lrqk_amd.engine import LightAttentionIndicesFactory as Engine
    gen = torch.Generator(device=DEV).manual_seed(l)

    def draw(heads, n):
        return torch.randn((batch, heads, n, d), generator=gen, device=DEV).to(dtype)
    engines = []
    for fill in (False, True):
        eng = Engine(num_lite_tokens=8, attn_topk=k, num_key_value_groups=hq // hkv, r=8, max_iter=2, tol=0.0, capacity=l + 64)
        eng.fill_victims, eng.victim_rows, eng.attn_in_step = fill, rows, True
        engines.append(eng)
    q, kk, vv = draw(hq, l), draw(hkv, l), draw(hkv, l)
    start = tuple(torch.randn((batch, hq, l, 8), generator=gen, device=DEV) for _ in range(2))
    for eng in engines:
        eng.init_factors = tuple(x.clone() for x in start)
        eng.prefill(q, kk, vv)
        eng.ws.victim_stats(reset=True)
    a, b = engines
    for step in range(12):   # (a flush of the ring among them)
        t = q[:, :, -1:] + 0.1 * draw(hq, 1), draw(hkv, 1), draw(hkv, 1)   # (near the prompt's last query)
        for eng in engines:
            eng.decode(*t)
        assert torch.equal(a._active_idx, b._active_idx) and torch.equal(a.last_attn, b.last_attn), step
        assert torch.equal(a.Kgpu, b.Kgpu) and torch.equal(a.Vgpu, b.Vgpu), step
    without, filled = (eng.ws.victim_stats() for eng in engines)
    print(f"rows over the host link: {without} without, {filled} with", flush=True)
    if d == 256:
        assert filled == without
    elif rows >= 96:   # (a few rows are replaced before they are asked for)
        assert filled < without


@pytest.mark.parametrize("dtype,batch,hq,hkv,d,l,k", [(torch.bfloat16, 3, 8, 2, 64, 1203, 128), (torch.float32, 2, 6, 3, 128, 901, 64),
                                                      (torch.bfloat16, 2, 4, 4, 128, 700, 96)])
def test_every_head_finds_its_rows_in_the_filled_cache(ops, dtype, batch, hq, hkv, d, l, k):
    """With the host store cleared behind a prompt, a row that enters the active set is its token's if it comes from the cache
    and zero if not: in the first step every head of every sequence has rows of the first kind, and none of a third."""
    from lrqk_amd.engine import LightAttentionIndicesFactory as Engine
    gen = torch.Generator(device=DEV).manual_seed(l)

    def draw(heads, n):
        return torch.randn((batch, heads, n, d), generator=gen, device=DEV).to(dtype)
    eng = Engine(num_lite_tokens=8, attn_topk=k, num_key_value_groups=hq // hkv, r=8, max_iter=2, tol=0.0, capacity=l + 64)
    eng.victim_rows, eng.attn_in_step = 512, True
    q, kk, vv = draw(hq, l), draw(hkv, l), draw(hkv, l)
    eng.init_factors = tuple(torch.randn((batch, hq, l, 8), generator=gen, device=DEV) for _ in range(2))
    eng.prefill(q, kk, vv)
    torch.cuda.synchronize()
    with torch.inference_mode():
        eng.KVcpu.data.zero_()
    before = eng._active_idx[:, :, :k].clone()
    eng.decode(q[:, :, -1:] + 0.1 * draw(hq, 1), draw(hkv, 1), draw(hkv, 1))
    after = eng._active_idx[:, :, :k]
    new = after != before
    ids = after.long().unsqueeze(-1).expand(-1, -1, -1, d)
    own = new
    for rows, got in ((kk, eng.Kgpu), (vv, eng.Vgpu)):
        got, want = got[:, :, :k], torch.gather(rows.repeat_interleave(hq // hkv, 1), 2, ids)
        same = (got == want).all(-1)
        assert (same | (new & (got == 0).all(-1))).all()
        own = own & same
    print(f"incoming rows per head: {new.sum(-1).tolist()}, from the cache: {own.sum(-1).tolist()}", flush=True)
    assert (own.sum(-1) > 0).all()


@pytest.mark.parametrize("engine,d,listed", [("plain", 8, True), ("switched off", 8, False), ("no hit miss", 8, False),
                                             ("staged fetch", 8, False), ("offload", 8, False), ("plain", 256, False)])
def test_a_prompt_lists_tokens_only_for_a_cache_that_it_fills(ops, monkeypatch, engine, d, listed):
    """The list of a prompt's next best tokens (128 heads x 1700: a block of its own) is given memory only where the prompt
    then fills the cache from it."""
    from lrqk_amd import engine as E
    kind = {"offload": E.LightAttentionIndicesOffloadPrefill, "no hit miss": E.LightAttentionIndicesNoHitMiss}
    eng = kind.get(engine, E.LightAttentionIndicesFactory)(num_lite_tokens=8, attn_topk=1700, num_key_value_groups=8, r=8,
                                                           max_iter=1, tol=0.0, capacity=2100)
    if engine == "switched off":
        eng.fill_victims = False
    if engine == "staged fetch":
        eng.fetch_mode = "staged"
    sizes, alloc = [], torch.cuda.caching_allocator_alloc

    def recorded(size, *a, **kw):
        sizes.append(size)
        return alloc(size, *a, **kw)
    gen = torch.Generator(device=DEV).manual_seed(d)
    q, k, v = (torch.randn((16, h, 2000, d), generator=gen, device=DEV) for h in (8, 1, 1))
    monkeypatch.setattr(torch.cuda, "caching_allocator_alloc", recorded)
    eng.prefill(q, k, v)
    need = 128 * 1701 * 4
    assert (need + need // 4 in sizes) == listed


def test_a_selection_that_failed_leaves_no_list(ops, monkeypatch):
    """A selection that raises before its kernels are launched (no memory for the score index) has listed nothing: nothing is
    put into the cache, which would take its 1.3 MB here."""
    gen = torch.Generator(device=DEV).manual_seed(1)
    a_k, q = (torch.randn((1, 4, n, 32), generator=gen, device=DEV) for n in (9000, 1))
    K, V = (torch.randn((1, 2, 9000, 64), generator=gen, device=DEV) for _ in range(2))
    ws = ops.Workspace()
    ws.victim_cache(512)
    ws.score_index(True)
    ops.score_select(ws, a_k, q, 9000, 300, list_next=True)
    want = ops.score_select(ws, a_k, q, 9000, 300)
    bigger = torch.cat([a_k, a_k], 2)
    sizes, alloc = [], torch.cuda.caching_allocator_alloc

    def refused(size, *a, **kw):
        sizes.append(size)
        if size > 1 << 20 and fails:
            raise torch.cuda.OutOfMemoryError("planted")
        return alloc(size, *a, **kw)
    monkeypatch.setattr(torch.cuda, "caching_allocator_alloc", refused)
    fails = True
    with pytest.raises(Exception, match="device memory"):
        ops.score_select(ws, bigger, q, 9000, 300, list_next=True)
    fails, sizes[:] = False, []
    ops.victim_fill(ws, K, V, 4, 9000)
    torch.cuda.synchronize()
    assert not sizes
    assert torch.equal(ops.score_select(ws, a_k, q, 9000, 300), want)


def test_an_index_whose_memory_was_had_in_part_is_dropped(ops, monkeypatch):
    """The rows of a larger index are there, its scales are not to be had: the selection raises, and the next one over the
    smaller factors, whose index went with the block that grew, indexes them again."""
    gen = torch.Generator(device=DEV).manual_seed(4)
    a_k, q = (torch.randn((1, 4, n, 16), generator=gen, device=DEV) for n in (9000, 1))
    bigger = torch.randn((1, 4, 120000, 16), generator=gen, device=DEV)
    ws = ops.Workspace()
    ws.score_index(True)
    want = ops.score_select(ws, a_k, q, 9000, 300)
    alloc, scales = torch.cuda.caching_allocator_alloc, 4 * 120000 * 2

    def refused(size, *a, **kw):
        if size == scales + scales // 4:
            raise torch.cuda.OutOfMemoryError("planted")
        return alloc(size, *a, **kw)
    with monkeypatch.context() as m:
        m.setattr(torch.cuda, "caching_allocator_alloc", refused)
        with pytest.raises(Exception, match=f"no {scales + scales // 4} bytes of device memory"):
            ops.score_select(ws, bigger, q, 120000, 300)
    for step in range(2):
        assert torch.equal(ops.score_select(ws, a_k, q, 9000, 300), want), step


@pytest.mark.parametrize("refused", ["rows", "positions"])
def test_a_prompt_does_not_fail_for_the_cache(ops, monkeypatch, refused):
    """Without memory for the victim cache (its rows; its position table) a prompt goes on, and the steps, for which there is
    memory again, are those after a prompt that does not fill it."""
    from lrqk_amd.engine import LightAttentionIndicesFactory as Engine
    gen = torch.Generator(device=DEV).manual_seed(3)

    def draw(heads, n):
        return torch.randn((1, heads, n, 64), generator=gen, device=DEV).to(torch.bfloat16)
    l, k, heads, capacity = 1200, 100, 8, 80000
    engines = [Engine(num_lite_tokens=8, attn_topk=k, num_key_value_groups=2, r=16, max_iter=1, tol=0.0, capacity=capacity)
               for _ in range(2)]
    prompt = draw(heads, l), draw(heads // 2, l), draw(heads // 2, l)
    start = tuple(torch.randn((1, heads, l, 16), generator=gen, device=DEV) for _ in range(2))
    rows = 1024
    need = {"rows": heads * rows * 16 * 16, "positions": (heads * rows + 3 * heads) * 4 + heads * capacity * 2 + 16}[refused]
    asked, alloc = [], torch.cuda.caching_allocator_alloc

    def without(size, *a, **kw):
        asked.append(size)
        if size == need + need // 4:
            raise torch.cuda.OutOfMemoryError("planted")
        return alloc(size, *a, **kw)
    for fill, eng in enumerate(engines):
        eng.fill_victims, eng.victim_rows, eng.attn_in_step, eng.init_factors = bool(fill), rows, True, start
        with monkeypatch.context() as m:
            m.setattr(torch.cuda, "caching_allocator_alloc", without)
            eng.prefill(*prompt)
    assert asked.count(need + need // 4) == 1
    for step in range(4):
        t = draw(heads, 1), draw(heads // 2, 1), draw(heads // 2, 1)
        for eng in engines:
            eng.decode(*t)
        assert torch.equal(engines[0]._active_idx, engines[1]._active_idx), step
        assert torch.equal(engines[0].last_attn, engines[1].last_attn), step


def test_a_captured_prompt_leaves_the_cache_alone(ops, monkeypatch):
    """Selection and fill in a graph: the cache is neither given memory nor taken for filled (every replay would fill it
    again, under the steps that use it); the same calls outside of it fill it."""
    gen = torch.Generator(device=DEV).manual_seed(2)
    a_k, q = (torch.randn((1, 4, n, 16), generator=gen, device=DEV) for n in (3000, 1))
    K, V = (torch.randn((1, 2, 3000, 64), generator=gen, device=DEV) for _ in range(2))
    ws, out = ops.Workspace(), torch.empty((1, 4, 300), dtype=torch.int32, device=DEV)
    ws.victim_cache(512)
    ops.score_select(ws, a_k, q, 3000, 300, out=out, list_next=True)   # (its workspace is there)
    want = out.clone()
    sizes, alloc = [], torch.cuda.caching_allocator_alloc

    def recorded(size, *a, **kw):
        sizes.append(size)
        return alloc(size, *a, **kw)
    monkeypatch.setattr(torch.cuda, "caching_allocator_alloc", recorded)

    def prompt():
        ops.score_select(ws, a_k, q, 3000, 300, out=out, list_next=True)
        ops.victim_fill(ws, K, V, 4, 3100)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        prompt()
    assert not sizes
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
    prompt()
    torch.cuda.synchronize()
    assert torch.equal(out, want) and 4 * 512 * 32 * 16 * 5 // 4 in sizes


@pytest.mark.parametrize("batch,hkv,l", [(1, 1, 300), (2, 3, 517), (1, 16, 1031)])
def test_prompt_rows_in_two_copies(ops, monkeypatch, batch, hkv, l):
    """A prompt whose first heads go ahead of the others (one head: a single copy; 6 and 16: pieces of 1 + 5, 2 + 14) is
    in the host store as given, also when the next prompt uses the same copy stream at once."""
    from lrqk_amd.engine import LightAttentionIndicesFactory as Engine
    monkeypatch.setattr(Engine, "_DMA_STORE_BYTES", 1)
    monkeypatch.setattr(Engine, "_DMA_PIECES_BYTES", 1)
    gen = torch.Generator(device=DEV).manual_seed(l)
    engines = []
    for _ in range(2):
        q, k, v = (torch.randn((batch, h, l, 64), generator=gen, device=DEV).to(torch.bfloat16) for h in (2 * hkv, hkv, hkv))
        eng = Engine(num_lite_tokens=8, attn_topk=64, num_key_value_groups=2, r=16, max_iter=1, tol=0.0, capacity=l + 9)
        eng.prefill(q, k, v)
        engines.append((eng, torch.cat([k, v], -1)))
    torch.cuda.current_stream().synchronize()
    for eng, want in engines:
        assert torch.equal(eng.KVcpu.tensor(), want.cpu())


@pytest.mark.parametrize("fails_at,first,second", [("als_prefill_store", 300, 260), ("als_prefill_store", 66, 300),
                                                   ("score_select", 300, 90)])
def test_a_prompt_that_failed_leaves_nothing_behind(ops, monkeypatch, fails_at, first, second):
    """An engine whose prefill raised takes the next prompt as a new one does: the same store, factors and steps past a
    flush of the ring."""
    from lrqk_amd.engine import LightAttentionIndicesFactory as Engine
    gen = torch.Generator(device=DEV).manual_seed(first)

    def rows(heads, n):
        return torch.randn((1, heads, n, 64), generator=gen, device=DEV).to(torch.bfloat16)
    lost = rows(4, first), rows(2, first), rows(2, first)
    prompt = rows(4, second), rows(2, second), rows(2, second)
    tokens = [(rows(4, 1), rows(2, 1), rows(2, 1)) for _ in range(20)]
    start = tuple(torch.randn((1, 4, second, 16), generator=gen, device=DEV) for _ in range(2))
    tried, fresh = (Engine(num_lite_tokens=8, attn_topk=64, num_key_value_groups=2, r=16, max_iter=2, tol=0.0, capacity=1200)
                    for _ in range(2))
    tried.init_factors = kept = tuple(torch.randn((1, 4, first, 16), generator=gen, device=DEV) for _ in range(2))

    def out_of_memory(*a, **kw):
        raise torch.cuda.OutOfMemoryError("planted")
    with monkeypatch.context() as m:
        m.setattr(ops, fails_at, out_of_memory)
        with pytest.raises(torch.cuda.OutOfMemoryError):
            tried.prefill(*lost)
    left = tried.init_factors
    for eng in (tried, fresh):
        eng.init_factors = start
        eng.prefill(*prompt)
        for t in tokens:
            eng.decode(*t)
    torch.cuda.synchronize()
    assert torch.equal(tried.KVcpu.tensor(), fresh.KVcpu.tensor())
    assert torch.equal(tried._A_K.data, fresh._A_K.data)
    assert torch.equal(tried.hit_indices, fresh.hit_indices) and torch.equal(tried.last_q_hat, fresh.last_q_hat)
    assert torch.equal(tried.Kgpu, fresh.Kgpu) and torch.equal(tried.Vgpu, fresh.Vgpu)
    assert left is kept
