"""GPU parity of the 16-byte forms of the layer's elementwise kernels where
they begin and end: RMSNorm rows around the chunk counts it is built for, rows
and tensors it leaves to the element-by-element form, and the FFN's gelu * up
over partial and several workgroups."""

import numpy as np
import pytest
import torch

import oracle as o
from helpers import down16, ulp_distance16, up16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [8, 100, 2048, 2056, 2560, 4096, 4104, 8192, 8200])
@pytest.mark.parametrize("offset", [0, 1])
def test_rms_norm_chunks(gpu, k, offset):
    """A mean square summed in fp32 in any order moves a row's norm by a few
    fp32 units: at most one unit of the 16-bit result, in few elements."""
    import sparkq

    m = 3
    print(f"[case] rms_norm k={k} offset={offset}", flush=True)
    for dtype in (o.BF16, o.F16):
        x = o.randn16(k, 1, m * k, 1.0, dtype).reshape(m, k)
        r = o.randn16(k, 2, m * k, 1.0, dtype).reshape(m, k)
        w = o.round16(1.0 + 0.2 * o.randn(k, 3, k), dtype)

        def place(a):
            t = up16(a, dtype, gpu)
            flat = torch.empty(t.numel() + offset, dtype=t.dtype, device=gpu)[offset:]
            return flat.copy_(t.reshape(-1)).view(t.shape)

        for res in (None, r):
            h = x if res is None else o.add16(x, r, dtype)
            n = sparkq.rms_norm(place(x), place(w), 1e-5,
                                residual=None if res is None else place(r))
            d = ulp_distance16(down16(n), o.rms_norm16(h, w, 1e-5, dtype), dtype)
            assert d.max() <= 1 and (d == 0).mean() > 0.98


def test_ffn_workspace_between_shapes(gpu):
    """Shapes whose projections need no workspace leave the counters of those
    that split along k alone: a prompt, a decoded token and the prompt again
    through one buffer give the prompt's output twice."""
    import sparkq
    from test_gpu_layer import _dev, _mat

    k, inter, g = 1024, 2560, 64
    ws = [_dev(_mat(7, s, n, kk, g, o.BF16), gpu, o.BF16)
          for s, n, kk in ((4, inter, k), (5, inter, k), (6, k, inter))]
    nw = up16(o.round16(np.ones(k, np.float32), o.BF16), o.BF16, gpu)

    def run(m):
        x = up16(o.randn16(m, 1, m * k).reshape(m, k), o.BF16, gpu)
        return sparkq.fused_ffn(x, x, nw, 1e-6, *ws, group_size=g)

    first = run(70)
    for m in (1, 2, 5, 16):
        run(m)
        print(f"[case] ffn workspace after m={m}", flush=True)
        assert torch.equal(run(70), first)


@pytest.mark.parametrize("m,inter", [(5, 64), (33, 2112), (40, 128), (129, 320)])
def test_gelu_chunks(gpu, m, inter):
    """act of the composed FFN equals the oracle's gelu(gate) * up of the
    device's own projections, and its output the down projection rounded, plus
    the residual, rounded again (in the bf16 GEMM's epilogue, over whole and
    split tiles), bit for bit."""
    import sparkq
    from test_gpu_layer import _dev, _mat, _plain

    k, g = 64, 32
    print(f"[case] gelu m={m} I={inter}", flush=True)
    for dtype in (o.BF16, o.F16):
        x = o.randn16(m, 1, m * k, 3.0, dtype).reshape(m, k)
        nw = o.round16(np.ones(k, np.float32), dtype)
        gate, up = (_mat(m, s, inter, k, g, dtype) for s in (4, 5))
        down = _mat(m, 6, k, inter, g, dtype)
        out, hid, nrm, act = (down16(t) for t in sparkq.fused_ffn(
            up16(x, dtype, gpu), up16(x[::-1].copy(), dtype, gpu), up16(nw, dtype, gpu), 1e-6,
            _dev(gate, gpu, dtype), _dev(up, gpu, dtype), _dev(down, gpu, dtype), group_size=g,
            return_intermediates=True))
        g16, u16 = (_plain(nrm, t, g, dtype, gpu) for t in (gate, up))
        assert np.array_equal(act, o.gelu_mul16(g16, u16, dtype))
        assert np.array_equal(out, o.add16(hid, _plain(act, down, g, dtype, gpu), dtype))


@pytest.mark.parametrize("m", [1, 5, 33])
def test_gelu_over_every_gate(gpu, m):
    """act of the FFN over every finite 16-bit gate (the division by 181/128
    is a product with its reciprocal in the kernels, and a division in the
    oracle), bit for bit, as the fused decode, the decode and the prefill
    projections feed it. Weight rows of scale 0 whose bias is the gate, and
    normed rows that are 1 once and 0 elsewhere, make the gates."""
    import sparkq
    from test_gpu_layer import _dev, _plain

    k, inter, g = 64, 65536, 64
    print(f"[case] every gate m={m}", flush=True)
    for dtype in (o.BF16, o.F16):
        bits = np.arange(inter, dtype=np.uint16)
        bits = np.where(np.isfinite(o.bits_to_f32(bits, dtype)), bits, 0).astype(np.uint16)
        one = o.round16(np.ones(1, np.float32), dtype)[0]
        codes, zero = np.zeros((inter, k // 8), np.uint32), np.zeros((inter, 1), np.uint16)
        gate = (codes, zero, bits[:, None].copy())
        up = (codes, zero, np.full((inter, 1), one, np.uint16))
        down = (np.zeros((k, inter // 8), np.uint32), np.zeros((k, inter // g), np.uint16),
                np.zeros((k, inter // g), np.uint16))
        x, nw = np.full((m, k), one, np.uint16), np.zeros(k, np.uint16)
        nw[0] = one
        zeros = up16(np.zeros((m, k), np.uint16), dtype, gpu)
        _, _, nrm, act = sparkq.fused_ffn(
            up16(x, dtype, gpu), zeros, up16(nw, dtype, gpu), 0.0, _dev(gate, gpu, dtype),
            _dev(up, gpu, dtype), _dev(down, gpu, dtype), group_size=g, return_intermediates=True)
        rows = np.tile(nw, (m, 1))
        g16, u16 = (_plain(rows, t, g, dtype, gpu) for t in (gate, up))
        assert (u16 == one).all()
        # (the sum with the scale's zero makes -0 a +0)
        for row in g16:
            assert np.array_equal(row, np.where(bits == 0x8000, 0, bits))
        got, ref = down16(act), o.gelu_mul16(g16, u16, dtype)
        assert np.array_equal(got, ref), int((got != ref).sum())
