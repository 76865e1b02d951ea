"""The scratch buffers behind the operators' workspaces (sparkq._lib). A HIP
graph replays with the addresses it was captured with, so a buffer that a
larger call outgrows must not go back to the allocator."""

import weakref

import pytest
import torch

from sparkq import _lib


@pytest.fixture
def host_buffers(monkeypatch):
    """workspace() on host memory, with tables of its own."""
    monkeypatch.setattr(_lib, "_raw_stream", lambda device: 0)
    monkeypatch.setattr(_lib, "_WS", {})
    monkeypatch.setattr(_lib, "_OUTGROWN", [], raising=False)
    return torch.device("cpu")


def test_outgrown_buffers_stay(host_buffers):
    refs, sizes = [], []
    for nbytes in (1000, 2 << 20, (2 << 20) + 1, 5 << 20, 9 << 20, 3 << 20):
        ptr, size = _lib.workspace(host_buffers, nbytes, "kind")
        buf = _lib._WS[(host_buffers.index, 0, "kind")]
        assert size >= nbytes and ptr.value == buf.data_ptr()
        assert not buf.any()
        if not refs or refs[-1]() is not buf:
            refs.append(weakref.ref(buf))
            sizes.append(size)
        del buf
    assert all(r() is not None for r in refs)
    # together the outgrown ones are smaller than the one in use
    assert sum(sizes[:-1]) < sizes[-1] == _lib.workspace(host_buffers, 1, "kind")[1]


def test_attention_workspace_fits_the_call():
    """fp32 queries and head dims of the vector kernel are not sized for the
    matrix-core kernel's splits."""
    lib = _lib.lib()
    call, any_call = (lib.sparkq_quantized_sdpa_call_workspace_bytes,
                      lib.sparkq_quantized_sdpa_workspace_bytes)
    shape = (1, 32, 8, 512, 4096)
    assert call(*shape, 128, 128, _lib.F32) == 0
    assert call(*shape, 160, 160, _lib.BF16) == 0
    assert call(*shape, 128, 64, _lib.BF16) == 0
    assert call(*shape, 128, 128, _lib.BF16) == any_call(*shape, 128) > 0
    assert call(1, 32, 8, 1, 4096, 128, 128, _lib.F32) > 0
    assert call(0, 32, 8, 1, 4096, 128, 128, _lib.F32) == 0


def _w4(gpu, m, n, k, g, seed):
    gen = torch.Generator().manual_seed(seed)
    x = torch.randn((m, k), generator=gen).to(torch.bfloat16).to(gpu)
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (n, k // 8), generator=gen, dtype=torch.int32).to(gpu)
    s = (torch.rand((n, k // g), generator=gen) * 0.01).to(torch.bfloat16).to(gpu)
    b = (torch.randn((n, k // g), generator=gen) * 0.05).to(torch.bfloat16).to(gpu)
    return x, w, s, b


def _w8(gpu, m, n, k, g, seed):
    x, w, s, b = _w4(gpu, m, n, k, g, seed)
    return x, torch.cat([w, w.flip(0)], 1), s, b


def test_calls_of_several_launches_share_no_scratch(monkeypatch):
    """Groupwise 8-bit and staged attention calls ask the allocator each time:
    two calls that are enqueued together hold different memory."""
    from sparkq import ext

    monkeypatch.setattr(_lib, "workspace", lambda *a: pytest.fail("shared workspace"))
    monkeypatch.setattr(_lib, "stream_handle", lambda device: None)
    monkeypatch.setattr(ext, "_require_device", lambda *a: None)
    held, live = [], []

    def scratch(device, nbytes):
        assert nbytes > 0
        live.append(torch.empty(nbytes, dtype=torch.uint8))
        return live[-1]

    def call(name, *args, device=None):
        held.append([a for a in args if a == live[-1].data_ptr()])

    monkeypatch.setattr(_lib, "scratch", scratch)
    monkeypatch.setattr(_lib, "call", call)
    cpu = torch.device("cpu")
    for seed in (1, 2):
        ext.affine_quantized_matmul(*_w8(cpu, 4, 256, 2560, 64, seed), group_size=64, bits=8)
        kv = (torch.zeros((1, 8, 900, 16), dtype=torch.int32),
              *(torch.zeros((1, 8, 900, 2), dtype=torch.bfloat16) for _ in range(2)))
        q = torch.zeros((1, 32, 4, 128), dtype=torch.bfloat16)
        ext.int8_quantized_sdpa(q, kv, kv, scale=1.0, group_size=64, bits=4, mask="causal")
    assert all(len(h) == 1 for h in held) and len({h[0] for h in held}) == 4


@pytest.mark.gpu
def test_threads_on_one_stream(gpu):
    """Two threads enqueue 8-bit calls on the same stream, interleaving their
    launches as they like: each gets its own result."""
    import threading

    import sparkq

    print("[case] two threads, one stream", flush=True)
    problems = [_w8(gpu, m, 1024, 2560, 64, m) for m in (8, 9)]
    call = lambda p: sparkq.affine_quantized_matmul(*p, group_size=64, bits=8)  # noqa: E731
    refs = [call(p) for p in problems]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        for _ in range(100):
            outs = [call(problems[i]) for _ in range(4)]
            if not all(torch.equal(y, refs[i]) for y in outs):
                bad.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


@pytest.mark.gpu
def test_two_graphs_on_one_capture_stream(gpu):
    """Graphs captured on one stream replay on two streams at once."""
    import sparkq

    print("[case] two graphs replayed side by side", flush=True)
    problems = [_w8(gpu, m, 1024, 2560, 64, m) for m in (8, 9)]
    refs = [sparkq.affine_quantized_matmul(*p, group_size=64, bits=8) for p in problems]
    outs = [torch.empty_like(r) for r in refs]
    torch.cuda.synchronize()
    side, graphs = torch.cuda.Stream(), []
    for p, y in zip(problems, outs):
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1], stream=side):
            for _ in range(10):
                sparkq.affine_quantized_matmul(*p, group_size=64, bits=8, out=y)
    streams = [torch.cuda.Stream() for _ in graphs]
    for replay in range(5):
        for y in outs:
            y.zero_()
        torch.cuda.synchronize()
        for graph, stream in zip(graphs, streams):
            with torch.cuda.stream(stream):
                graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(y, r) for y, r in zip(outs, refs)), replay


@pytest.mark.gpu
@pytest.mark.parametrize("bits", [4, 8])
def test_graph_survives_a_larger_call(gpu, bits):
    """Capture a small call after a warm-up on its stream, run a larger one
    there, fill what the allocator then hands out, and replay: the output is
    the eager one and the new memory is as it was."""
    import sparkq

    print(f"[case] workspace growth under a graph, {bits}-bit", flush=True)
    g = 64

    def problem(m, n, k, seed):
        return (_w4 if bits == 4 else _w8)(gpu, m, n, k, g, seed)

    small, large = problem(48, 512, 2560, 1), problem(900, 3584, 2560, 2)
    out = torch.empty((48, 512), dtype=torch.bfloat16, device=gpu)

    def call(args, out=None):
        return sparkq.affine_quantized_matmul(*args, group_size=g, bits=bits, out=out)

    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        call(small, out)
        eager = out.clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        call(small, out)
    with torch.cuda.stream(stream):
        big = call(large).clone()
        canaries = [torch.full((size,), 0x5A, dtype=torch.uint8, device=gpu)
                    for size in (1 << 12, 1 << 16, 1 << 20, 1 << 21, 1 << 22, 1 << 23)]
    torch.cuda.synchronize()
    for replay in range(3):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), replay
        assert all(bool((c == 0x5A).all()) for c in canaries), replay
        with torch.cuda.stream(stream):
            assert torch.equal(call(large), big)
        torch.cuda.synchronize()
