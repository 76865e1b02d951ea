"""GPU parity of the matrix-core staged attention (sdpa_stage_kernel: 16-bit
queries, one head dim of 64/96/128/256) where its tiles and splits end: row
counts around 128-row tiles, contexts around 32-token blocks, every (head
dim, group size) it is built for, rows that see nothing, a token-strided
cache view, and calls it leaves to the vector kernel. The bound is that of
fp32 arithmetic: the products are exact, so what remains are the fp32 sums
over at most a few thousand terms (1e-5 of the result's norm)."""

import math

import numpy as np
import pytest
import torch

import oracle as o
from helpers import up16
from test_gpu_sdpa_staged import _cache

pytestmark = pytest.mark.gpu

CASES = [
    # b, hq, hkv, L, n, d, g, bits, qdtype, mask
    (1, 4, 1, 31, 31, 64, 32, 2, o.BF16, "causal"),     # 124 rows, one short block
    (1, 4, 1, 32, 32, 64, 64, 4, o.F16, "causal"),      # exactly one tile, one block
    (2, 3, 1, 43, 65, 96, 32, 8, o.BF16, "causal"),     # 129 rows, a token past two blocks
    (1, 6, 2, 2, 33, 128, 32, 4, o.F16, None),          # six rows of 128
    (1, 8, 2, 1, 257, 128, 128, 2, o.BF16, "bool"),     # one query token, a mask array
    (1, 4, 2, 33, 700, 128, 64, 8, o.F16, "add"),
    (1, 4, 4, 130, 131, 256, 32, 4, o.BF16, "bool"),
    (1, 4, 2, 65, 300, 256, 64, 2, o.F16, "causal"),
    (1, 2, 1, 70, 90, 256, 128, 8, o.BF16, "add"),
    (1, 6, 2, 9, 5, 96, 32, 4, o.BF16, "causal"),       # L > N: rows that see nothing
    (1, 10, 2, 300, 2100, 128, 64, 4, o.BF16, "causal"),  # several tiles and splits
]


@pytest.mark.parametrize("b,hq,hkv,length,n,d,g,bits,qdtype,mask", CASES)
def test_stage_kernel_matches_oracle(gpu, b, hq, hkv, length, n, d, g, bits, qdtype, mask):
    import sparkq

    print(f"[case] stage b={b} hq={hq} hkv={hkv} L={length} N={n} D={d} G={g} bits={bits} "
          f"q={qdtype} mask={mask}", flush=True)
    seed = n + d + bits + length
    (kt, kd), (vt, vd) = (_cache(gpu, b, hkv, n, d, g, bits, qdtype, seed + i) for i in (0, 1))
    q16 = o.round16(o.randn(seed, 72, b * hq * length * d).reshape(b, hq, length, d), qdtype)
    rng = np.random.default_rng(seed)
    mask_t = mask_ref = mask
    if mask == "bool":
        m = rng.random((hq, length, n)) > 0.4
        if length > 1:
            m[:, 0] = False
        mask_t, mask_ref = torch.from_numpy(m).to(gpu), m[None]
    elif mask == "add":
        m = (rng.standard_normal((1, 1, length, n)) * 2).astype(np.float32)
        m[..., : n // 2] = -np.inf
        mask_t, mask_ref = torch.from_numpy(m).to(gpu), m
    scale = 1.0 / math.sqrt(d)
    qt = up16(q16, qdtype, gpu)

    def attend(kt, vt):
        return sparkq.ext.staged_quantized_sdpa(qt, kt, vt, scale=scale, group_size=g, bits=bits,
                                                mask=mask_t, out_dtype=torch.float32)

    y = attend(kt, vt).cpu().numpy()
    ref = o.sdpa_staged(o.bits_to_f32(q16, qdtype), kd, vd, scale, mask_ref, qdtype)
    rel = np.linalg.norm(y - ref) / np.linalg.norm(ref)
    print(f"rel {rel:.2e}", flush=True)
    assert np.isfinite(y).all() and rel <= 1e-5
    # the same tokens behind a cache of a larger capacity give the same bits,
    # and a query that is not 16-byte aligned (the vector kernel) the same values
    def room(t):
        big = torch.full((t.shape[0], t.shape[1], n + 7, t.shape[3]), 1, dtype=t.dtype, device=gpu)
        big[:, :, :n] = t
        return big[:, :, :n]

    wide = attend(tuple(room(t) for t in kt), tuple(room(t) for t in vt)).cpu().numpy()
    assert np.array_equal(wide, y)
    flat = torch.empty(qt.numel() + 1, dtype=qt.dtype, device=gpu)[1:]
    flat.copy_(qt.reshape(-1))
    qt = flat.view(qt.shape)
    rel = np.linalg.norm(attend(kt, vt).cpu().numpy() - ref) / np.linalg.norm(ref)
    assert rel <= 1e-5


def test_stage_takes_a_smaller_workspace(gpu):
    """A C caller may give less than the matrix-core kernel's splits use, down
    to what the vector kernel needs (nothing here): it then runs fewer. Less
    than that is refused."""
    import ctypes

    from sparkq import _lib

    print("[case] stage with a small workspace", flush=True)
    hq, hkv, length, n, d, g, bits = 32, 8, 200, 900, 128, 64, 4
    (kt, _), (vt, _) = (_cache(gpu, 1, hkv, n, d, g, bits, o.BF16, i) for i in (0, 1))
    qt = up16(o.randn16(4, 72, hq * length * d).reshape(1, hq, length, d), o.BF16, gpu)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    ng = d // g
    strides = (ctypes.c_int64 * 12)(*(2 * [hkv * n * d // 2, n * d // 2, d // 2,
                                           hkv * n * ng, n * ng, ng]))

    def attend(nbytes, rows=length):
        ws = torch.empty(nbytes, dtype=torch.uint8, device=gpu) if nbytes else None
        y = torch.full((1, hq, rows, d), float("nan"), dtype=torch.float32, device=gpu)
        q = qt[:, :, :rows].contiguous()
        rc = _lib.lib().sparkq_quantized_sdpa(
            ptr(q), *map(ptr, kt), *map(ptr, vt), None, 1, _lib.F32, None, ptr(y), 1, hq, hkv,
            rows, n, d, d, g, bits, _lib.BF16, _lib.F32, d ** -0.5, strides,
            ptr(ws) if nbytes else None, nbytes, _lib.stream_handle(gpu))
        torch.cuda.synchronize()
        return rc, y

    query = _lib.lib().sparkq_quantized_sdpa_call_workspace_bytes
    full = query(1, hq, hkv, length, n, d, d, _lib.BF16)
    assert full > query(1, hq, hkv, length, n, d, d, _lib.F32) == 0
    rc, ref = attend(full)
    assert rc == 0
    for nbytes in (full - 1, full // 2, 4096, 0):
        rc, y = attend(nbytes)
        assert rc == 0, (nbytes, _lib.lib().sparkq_last_error())
        assert float((y - ref).norm()) <= 1e-5 * float(ref.norm()), nbytes
    # one row: the vector kernel splits too, and its need is the least
    least = query(1, hq, hkv, 1, n, d, d, _lib.F32)
    assert least > 0
    assert attend(least, 1)[0] == 0
    assert attend(least - 1, 1)[0] == _lib.ERR_WORKSPACE
