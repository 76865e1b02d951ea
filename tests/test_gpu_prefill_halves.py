"""Causal prefill over an 8-bit affine cache at head dim 256 with one to two
row tiles per CU: tiles in halves against whole tiles and the float64 oracle.
The halves' weights are the whole tile's (powers of two apart) and their sums
fp32: 1e-5 of the result's norm."""

import math

import numpy as np
import pytest
import torch

import oracle as o
from helpers import up16
from test_gpu_sdpa_staged import _cache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,hq,hkv,length,n,qdtype", [
    (2, 64, 32, 300, 300, o.BF16),   # 320 tiles, the last of 88 rows
    (1, 32, 32, 1030, 1100, o.F16),  # 288 tiles, a context past the queries
    (4, 64, 64, 100, 150, o.BF16),   # 256 tiles of 100 rows, N at the bound
    (4, 64, 64, 100, 151, o.BF16),   # one token past it: whole tiles
])
def test_causal_halves(gpu, b, hq, hkv, length, n, qdtype, monkeypatch):
    import sparkq

    d, g = 256, 32
    print(f"[case] halves b={b} {hq}/{hkv} L={length} N={n} q={qdtype}", flush=True)
    (kt, kd), (vt, vd) = (_cache(gpu, b, hkv, n, d, g, 8, qdtype, n + i) for i in (0, 1))
    q16 = o.round16(o.randn(n, 72, b * hq * length * d).reshape(b, hq, length, d), qdtype)
    qt = up16(q16, qdtype, gpu)

    def attend():
        # halves are what the planner chose, or not
        need = sparkq._lib.lib().sparkq_int8kv_sdpa_prefill_affine_workspace_bytes(
            b, hq, hkv, length, n, d, 1)
        assert (need > 0) == halves
        return sparkq.int8_quantized_sdpa(qt, kt, vt, scale=1 / math.sqrt(d), group_size=g, bits=8,
                                          mask="causal", out_dtype=torch.float32)

    # (forced: the planner takes prompts of 2048 tokens and more)
    monkeypatch.setenv("SPARKQ_PREFILL_HALVES", "1")
    halves = 2 * n <= 3 * length
    y = attend()
    assert torch.equal(attend(), y)
    monkeypatch.setenv("SPARKQ_PREFILL_NO_HALVES", "1")
    halves = False
    whole = attend()
    rel = float((y - whole).norm() / whole.norm())
    print(f"halves against whole {rel:.2e}", flush=True)
    assert rel <= 1e-5
    # the oracle on the first and last heads (the rounded weights of 16 bits
    # leave 2^-9 or 2^-12 of each)
    ratio = hq // hkv
    for h in (0, hq - 1):
        ref = o.sdpa_staged(o.bits_to_f32(q16[-1:, h:h + 1], qdtype), kd[-1:, h // ratio:h // ratio + 1],
                            vd[-1:, h // ratio:h // ratio + 1], 1 / math.sqrt(d), "causal", qdtype)
        got = y[-1:, h:h + 1].cpu().numpy()
        assert np.linalg.norm(got - ref) <= 4e-3 * np.linalg.norm(ref)


def test_halves_without_a_workspace(gpu, monkeypatch):
    """A C caller that passes none gets whole tiles, the same bits as with the
    halves switched off."""
    import ctypes

    import sparkq
    from sparkq import _lib

    b, h, length, d, g = 4, 64, 100, 256, 32
    print("[case] halves without a workspace", flush=True)
    monkeypatch.setenv("SPARKQ_PREFILL_HALVES", "1")
    (kt, _), (vt, _) = (_cache(gpu, b, h, length, d, g, 8, o.BF16, i) for i in (0, 1))
    qt = up16(o.randn16(3, 72, b * h * length * d).reshape(b, h, length, d), o.BF16, gpu)
    y = torch.empty_like(qt)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    strides = (ctypes.c_int64 * 12)(*(2 * [h * length * d, length * d, d, h * length * (d // g),
                                           length * (d // g), d // g]))
    rc = _lib.lib().sparkq_int8kv_sdpa_prefill_affine(
        ptr(qt), *map(ptr, kt), *map(ptr, vt), ptr(y), b, h, h, length, length, d, g, 1,
        _lib.BF16, _lib.BF16, 0.0625, strides, None, 0, _lib.stream_handle(gpu))
    assert rc == 0, _lib.lib().sparkq_last_error()
    monkeypatch.setenv("SPARKQ_PREFILL_NO_HALVES", "1")
    whole = sparkq.int8_quantized_sdpa(qt, kt, vt, scale=0.0625, group_size=g, bits=8,
                                       mask="causal")
    assert torch.equal(y, whole)
