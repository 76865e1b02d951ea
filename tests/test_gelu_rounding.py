"""The division of the 16-bit gelu by 181/128 against the product with its
fp32 reciprocal, over every finite gate of both 16-bit types: the same 16 bits
after rounding, as the comment at gelu_mul argues. This checks the argument in
numpy; test_gpu_layer_chunks.py runs the kernels over the same gates."""

import numpy as np
import pytest
import torch


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gelu_reciprocal_rounds_as_the_division(dtype):
    bits = torch.from_numpy(np.arange(65536, dtype=np.uint16).view(np.int16))
    gate = bits.view(dtype).float().numpy()
    c = np.float32(1.4140625)
    with np.errstate(all="ignore"):
        div, mul = gate / c, gate * (np.float32(1.0) / c)
    a, b = (torch.from_numpy(v).to(dtype) for v in (div, mul))
    ok = ~torch.isnan(a)
    assert torch.equal(torch.isnan(a), torch.isnan(b))
    assert torch.equal(a[ok].view(torch.int16), b[ok].view(torch.int16))
