"""The per-stream buffers of the launch path: what a captured graph was given stays valid, and what no graph can hold
goes back to the allocator."""

import weakref

import pytest
import torch


@pytest.fixture
def hip(monkeypatch):
    """The buffer code on CPU tensors, as one stream of one device sees it; hip.capture is the stream's capture id."""
    from bitexact import _hip

    class Lib:
        capture = 0

        def bx_capture_id(self, stream):
            return self.capture
    fake = Lib()
    for name in ("_ws", "_ws_graph", "_tmp"):
        monkeypatch.setattr(_hip, name, {}, raising=False)
    monkeypatch.setattr(_hip, "_ws_outgrown", [], raising=False)
    monkeypatch.setattr(_hip, "_raw_stream", lambda i: 7)
    monkeypatch.setattr(_hip, "lib", lambda: fake)
    return _hip, fake, torch.device("cpu", 0)


def test_outgrown_workspace_stays_alive(hip):
    _hip, _, dev = hip
    first = weakref.ref(_hip.workspace(dev, 100)[0])
    n = first().numel()
    big, size = _hip.workspace(dev, n + 1)
    assert first() is not None and big is not first() and size >= 2 * n and not big.any()
    assert _hip.workspace(dev, 1)[0] is big


def test_small_scratch_is_never_replaced_and_large_is_not_kept(hip):
    _hip, _, dev = hip
    small = _hip.scratch(dev, 100)[0]
    large, n = _hip.scratch(dev, (8 << 20) + 1)
    assert n > 8 << 20 and large is not small
    large = weakref.ref(large)
    assert large() is None, "large scratch outlives its call"
    assert _hip.scratch(dev, 1 << 20)[0] is small and _hip.scratch(dev, 8 << 20)[0] is small


def test_workspace_made_in_a_capture_stays_with_it(hip):
    _hip, lib, dev = hip
    eager = _hip.workspace(dev, 100)[0]
    lib.capture = 3
    assert _hip.workspace(dev, 100)[0] is eager
    own = _hip.workspace(dev, 5 << 20)[0]
    assert _hip.workspace(dev, 4 << 20)[0] is own and _hip.workspace(dev, 100)[0] is eager
    lib.capture = 4
    other = _hip.workspace(dev, 5 << 20)[0]
    assert other is not own
    lib.capture = 0
    later = _hip.workspace(dev, 5 << 20)[0]
    assert later is not own and later is not other


@pytest.mark.gpu
@pytest.mark.parametrize("warm", [True, False])
def test_graph_outlives_larger_calls(dev, warm):
    """Long-context attention and a split linear captured at a small batch; then larger eager calls on the capture
    stream and another capture there (whose graph runs first), and tensors that take up whatever memory was given
    back. Replays of the first graph give the eager result and leave those tensors alone. warm: the calls ran on the
    stream before the capture (its buffers are there already) or not (they come from the graph)."""
    from bitexact.exact.consts import decompose, exp2_table
    from bitexact.vllm_plugin import tri_exact_attn, tri_paged
    from bitexact.vllm_plugin.exact_gemm import exact_linear
    g = torch.Generator().manual_seed(5)
    HD, HKV, M, bs, keys = 64, 8, 4, 16, 2304
    nblk, top = keys // bs, 24
    cache = tri_paged.to_limbs((torch.randn(nblk, HKV, bs, 2 * HD, generator=g) * 2 ** 18).to(torch.int32).to(dev))
    lut = exp2_table(dev)
    dec = decompose((torch.randn(512, 2048, generator=g) * 0.02).to(torch.bfloat16).to(dev))

    def step(R):
        h = torch.Generator().manual_seed(R)
        bt = torch.stack([torch.randperm(nblk, generator=h) for _ in range(R)]).to(torch.int32).to(dev)
        q = torch.randint(-(1 << 22), 1 << 22, (R, HKV, M, HD), generator=h).to(torch.int32).to(dev)
        sh = torch.full((R, HKV, M), -22, device=dev)
        qpos = torch.randint(keys // 2, keys, (R, 1), generator=h).expand(R, M).contiguous().to(dev)
        rmap = torch.arange(R, device=dev)
        rows = torch.randint(-(1 << 22), 1 << 22, (40 * R, 2048), generator=h).to(torch.int32).to(dev)
        shr, flag = torch.full((40 * R,), -22, device=dev), torch.zeros(1, dtype=torch.int32, device=dev)

        def run():
            n, d = tri_exact_attn.attend(q, sh, qpos, cache, bt, rmap, lut, 387270501)
            y = exact_linear(rows, shr, dec["limbs"], dec["d"], dec["g"], dec["ell_cnt"], dec["ell_col"],
                             dec["ell_val"], dec["R"], flag, False)
            return n, d, y
        return run
    same = lambda a, b: all(torch.equal(x, y) for x, y in zip(a, b))
    small, large = step(8), step(top)
    ref, ref_large = small(), large()
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()

    def capture(run):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            out = run()
        return graph, out
    if warm:
        with torch.cuda.stream(stream):
            small()
        torch.cuda.synchronize()
    graph, out = capture(small)
    graph2, out2 = capture(large)
    with torch.cuda.stream(stream):
        eager = large()
    torch.cuda.synchronize()
    assert same(eager, ref_large)
    graph2.replay()
    torch.cuda.synchronize()
    assert same(out2, ref_large)
    torch.cuda.empty_cache()
    taken = [torch.full((n << 20,), 7, dtype=torch.uint8, device=dev) for n in (1, 1, 2, 4, 8, 16, 32, 64)]
    with torch.cuda.stream(stream):
        taken += [torch.full((n << 20,), 7, dtype=torch.uint8, device=dev) for n in (1, 1, 2, 4, 8, 16, 32, 64)]
    torch.cuda.synchronize()
    for _ in range(3):
        for t in out:
            t.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        assert same(out, ref)
        assert same(small(), ref)
    assert all(bool((t == 7).all()) for t in taken)
