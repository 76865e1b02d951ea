"""GPU parity of the affine prefill GEMM (affine_gemm_kernel: 4-bit weights of
float16 activations from 33 rows, 8-bit weights) where its tiles,
units of 128 k and pieces end, for every (width, group size, type) it
is built for, against the float64 oracle. Products are exact and every sum is
fp32; the terms s*q and b cancel to a few times the result's size: 1e-5 of
its norm. The pieces are forced, so that short K splits too."""

import numpy as np
import pytest
import torch

import oracle as o
from helpers import down16, rel_l2, up16, up32, w4_problem
from test_gpu_w8_affine import _dev_scales, _problem

pytestmark = pytest.mark.gpu

W4 = [
    # m, n, k, g, pieces (0: the plan's)
    (33, 1, 64, 32, 1), (64, 127, 192, 64, 1), (65, 129, 128, 128, 1), (129, 257, 1088, 32, 3),
    (40, 512, 1280, 64, 8), (600, 130, 640, 128, 5), (64, 260, 320, 32, 2),
    (333, 384, 9728, 128, 0), (577, 1025, 704, 64, 0),
]
W8 = [
    (1, 130, 64, 32, o.BF16, o.BF16, 1), (3, 512, 2560, 64, o.F16, o.F16, 0),
    (64, 1, 32, 32, o.BF16, o.BF16, 1), (65, 129, 96, 32, o.F16, o.F32, 1),
    (127, 127, 160, 32, o.BF16, o.F32, 2), (130, 300, 1216, 64, o.F16, o.F16, 4),
    (64, 257, 640, 128, o.BF16, o.BF16, 5), (200, 130, 384, 128, o.F16, o.BF16, 1),
    (513, 640, 2560, 64, o.BF16, o.F32, 0), (70, 130, 192, 64, o.BF16, o.F16, 1),
]


def _force(monkeypatch, s):
    if s:
        monkeypatch.setenv("SPARKQ_AFFG_S", str(s))


@pytest.mark.parametrize("m,n,k,g,s", W4)
def test_w4_f16_prefill(gpu, m, n, k, g, s, monkeypatch):
    import sparkq

    print(f"[case] affgemm w4 m={m} n={n} k={k} g={g} s={s}", flush=True)
    _force(monkeypatch, s)
    x, wq, sc, b = w4_problem(m, n, k, g, o.F16, seed=m + n)
    args = (up16(x, o.F16, gpu), up32(wq, gpu), up16(sc, o.F16, gpu), up16(b, o.F16, gpu))
    ref = o.w4a16_matmul(x, wq, sc, b, g, o.F16)
    y = sparkq.affine_quantized_matmul(*args, group_size=g, out_dtype=torch.float32)
    rel = rel_l2(y.cpu().numpy(), ref)
    print(f"rel {rel:.2e}", flush=True)
    assert rel <= 1e-5
    y16 = sparkq.affine_quantized_matmul(*args, group_size=g)
    assert torch.equal(y16, y.to(torch.float16))


@pytest.mark.parametrize("m,n,k,g,dtype,sdtype,s", W8)
def test_w8_prefill(gpu, m, n, k, g, dtype, sdtype, s, monkeypatch):
    import sparkq

    print(f"[case] affgemm w8 m={m} n={n} k={k} g={g} x={dtype} s={sdtype} pieces={s}", flush=True)
    _force(monkeypatch, s)
    x, words, sc, b = _problem(m, n, k, g, dtype, sdtype, seed=m + n)
    args = (up16(x, dtype, gpu), up32(words, gpu), _dev_scales(sc, sdtype, gpu),
            _dev_scales(b, sdtype, gpu))
    ref = o.w8_affine_matmul(x, words, sc, b, g, dtype, sdtype)
    y = sparkq.affine_quantized_matmul(*args, group_size=g, bits=8, out_dtype=torch.float32)
    rel = rel_l2(y.cpu().numpy(), ref)
    print(f"rel {rel:.2e}", flush=True)
    assert rel <= 1e-5
    # the kernel that needs no workspace gives the same to fp32 sums
    monkeypatch.setenv("SPARKQ_W8AFF_GEMM_FROM", "1000000")
    z = sparkq.affine_quantized_matmul(*args, group_size=g, bits=8, out_dtype=torch.float32)
    assert rel_l2(y.cpu().numpy(), z.cpu().numpy()) <= 1e-5


def _shifted(x, dtype, mean):
    return o.round16(o.bits_to_f32(x, dtype) + np.float32(mean), dtype)


@pytest.mark.parametrize("mean", [0.0, 1.0])
@pytest.mark.parametrize("bits,m,n,k,g,dtype,sdtype,s", [
    (4, 40, 128, 9728, 32, o.F16, o.F16, 1), (4, 64, 200, 9728, 64, o.F16, o.F16, 3),
    (4, 33, 130, 9728, 128, o.F16, o.F16, 0), (4, 96, 256, 2624, 64, o.F16, o.F16, 1),
    (8, 1, 512, 9728, 64, o.BF16, o.F32, 1), (8, 40, 128, 9728, 64, o.BF16, o.F32, 1),
    (8, 64, 256, 2560, 64, o.BF16, o.BF16, 3), (8, 64, 200, 9728, 128, o.F16, o.F16, 1),
    (8, 40, 130, 9728, 32, o.F16, o.F16, 1), (8, 33, 128, 2592, 32, o.BF16, o.F32, 0),
])
def test_error_over_long_rows(gpu, bits, m, n, k, g, dtype, sdtype, s, mean, monkeypatch):
    """Long rows, and activations of mean 1, where the scale and bias parts
    cancel. Each group rounds the running sum twice, by at most 2^-24 of it;
    2 K/G roundings add in quadrature."""
    import sparkq

    print(f"[case] affgemm err w{bits} m={m} n={n} k={k} g={g} mean={mean}", flush=True)
    _force(monkeypatch, s)
    if bits == 4:
        x, words, sc, b = w4_problem(m, n, k, g, dtype, seed=m + n)
    else:
        x, words, sc, b = _problem(m, n, k, g, dtype, sdtype, seed=m + n)
    x = _shifted(x, dtype, mean)
    ref = (o.w4a16_matmul(x, words, sc, b, g, dtype) if bits == 4
           else o.w8_affine_matmul(x, words, sc, b, g, dtype, sdtype))
    y = sparkq.affine_quantized_matmul(up16(x, dtype, gpu), up32(words, gpu),
                                       _dev_scales(sc, sdtype, gpu), _dev_scales(b, sdtype, gpu),
                                       group_size=g, bits=bits, out_dtype=torch.float32)
    rel = rel_l2(y.cpu().numpy(), ref)
    bound = (2 * k / g) ** 0.5 * 2.0 ** -24
    print(f"rel {rel:.2e} bound {bound:.2e}", flush=True)
    assert rel <= bound


@pytest.mark.parametrize("m,n,k,g", [(1, 130, 64, 64), (33, 200, 320, 64), (40, 130, 96, 32),
                                     (2, 300, 256, 128), (257, 4096, 320, 64), (5, 70, 384, 64)])
def test_w8_short_rows_on_both_kernels(gpu, m, n, k, g, monkeypatch):
    """Around the rule that keeps short rows in one launch: the planned kernel
    and each of the two agree with the oracle."""
    import sparkq

    print(f"[case] affgemm w8 short m={m} n={n} k={k} g={g}", flush=True)
    x, words, sc, b = _problem(m, n, k, g, o.BF16, o.F32, seed=m + n)
    args = (up16(x, o.BF16, gpu), up32(words, gpu), _dev_scales(sc, o.F32, gpu),
            _dev_scales(b, o.F32, gpu))
    ref = o.w8_affine_matmul(x, words, sc, b, g, o.BF16, o.F32)
    for route in (None, "1", "1000000"):
        if route is not None:
            monkeypatch.setenv("SPARKQ_W8AFF_GEMM_FROM", route)
        y = sparkq.affine_quantized_matmul(*args, group_size=g, bits=8)
        assert rel_l2(y.cpu().numpy(), ref) <= 1e-6, route
