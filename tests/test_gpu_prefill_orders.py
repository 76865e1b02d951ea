"""The affine prefill's chunks and work orders: eight, four and two chunks per
tile and whole tiles at every head dim, in runs and dealt over the XCDs. The
order of the work changes no sum, so any order gives the same bits as the plain
one; one head is checked against the float64 oracle."""

import math

import numpy as np
import pytest
import torch

import oracle as o
from helpers import up16
from test_gpu_sdpa_staged import _cache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,hq,hkv,length,n,qdtype", [
    (256, 16, 4, 8, 300, o.BF16),      # eight chunks, runs
    (256, 16, 4, 512, 700, o.F16),     # four
    (256, 16, 4, 1000, 1000, o.BF16),  # two chunks on 250 CUs
    (256, 16, 4, 1216, 1216, o.BF16),  # two chunks, dealt
    (256, 16, 4, 2112, 3300, o.BF16),  # whole tiles, dealt
    (128, 32, 8, 40, 260, o.BF16),     # eight chunks, own sums in registers
    (128, 32, 8, 512, 512, o.F16),     # two
    (64, 16, 4, 100, 400, o.BF16),     # eight
    (64, 16, 4, 1000, 1001, o.F16),    # two
])
def test_orders_give_the_same_bits(gpu, d, hq, hkv, length, n, qdtype, monkeypatch):
    import sparkq

    g = 32
    print(f"[case] prefill order d={d} {hq}/{hkv} L={length} N={n}", flush=True)
    (kt, kd), (vt, vd) = (_cache(gpu, 1, hkv, n, d, g, 8, qdtype, n + i) for i in (0, 1))
    q16 = o.round16(o.randn(n, 73, hq * length * d).reshape(1, hq, length, d), qdtype)
    qt = up16(q16, qdtype, gpu)

    def attend():
        return sparkq.int8_quantized_sdpa(qt, kt, vt, scale=1 / math.sqrt(d), group_size=g, bits=8,
                                          mask="causal", out_dtype=torch.float32)

    y = attend()
    monkeypatch.setenv("SPARKQ_PREFILL_NO_XCD", "1")
    assert torch.equal(attend(), y)
    h = hq - 1
    ref = o.sdpa_staged(o.bits_to_f32(q16[:, h:], qdtype), kd[:, -1:], vd[:, -1:],
                        1 / math.sqrt(d), "causal", qdtype)
    got = y[:, h:].cpu().numpy()
    # (the weights are rounded to 16 bits: 2^-9 or 2^-12 of each)
    assert np.linalg.norm(got - ref) <= 4e-3 * np.linalg.norm(ref)
