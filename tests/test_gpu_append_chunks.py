"""The 16-byte quantize-on-append against the thread-per-group kernel, byte
for byte: every width and group size, head dims around them, remainders of the
workgroup, a strided cache at an odd offset, and groups whose values decide
the order of the comparisons (zeros of both signs, infinities, NaN first and
later, constants)."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [8, 4, 2])
@pytest.mark.parametrize("b,h,length,d,g", [(1, 1, 1, 32, 32), (2, 3, 7, 96, 32), (1, 4, 33, 128, 128),
                                            (1, 2, 65, 256, 64), (1, 5, 3, 320, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_append_chunks_equal_thread_kernel(gpu, bits, b, h, length, d, g, dtype, monkeypatch):
    import sparkq

    print(f"[case] append bits={bits} {b}x{h}x{length}x{d} G={g} {dtype}", flush=True)
    gen = torch.Generator().manual_seed(d + length)
    x = torch.randn((b, h, length, d), generator=gen)
    flat = x.view(-1, g)
    special = [0.0, -0.0, 1.5, -2.0, np.inf, -np.inf, np.nan]
    for i in range(0, flat.shape[0], 3):  # a third of the groups
        pick = torch.randint(0, 4 + i % 4, (g,), generator=gen)
        flat[i] = torch.tensor(special)[pick]
        if i % 2:
            flat[i] = flat[i, 0]
    x = x.to(dtype).to(gpu)

    def cache():
        room = length + 9
        return (torch.full((b, h, room, d * bits // 32), 7, dtype=torch.int32, device=gpu),
                torch.full((b, h, room, d // g), 3, dtype=dtype, device=gpu),
                torch.full((b, h, room, d // g), 5, dtype=dtype, device=gpu))

    got, want = cache(), cache()
    sparkq.kv_append(x, got, 5, group_size=g, bits=bits)
    monkeypatch.setenv("SPARKQ_KV_APPEND_THREAD", "1")
    sparkq.kv_append(x, want, 5, group_size=g, bits=bits)
    assert torch.equal(got[0], want[0])
    for p, q in zip(got[1:], want[1:]):
        nan = torch.isnan(q)
        assert torch.equal(torch.isnan(p), nan)
        assert torch.equal(p.view(torch.int16)[~nan], q.view(torch.int16)[~nan])
