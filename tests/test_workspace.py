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
        x, w, s, b = _w4(gpu, m, n, k, g, seed)
        if bits == 8:
            w = torch.cat([w, w.flip(0)], 1)
        return x, w, s, b

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
