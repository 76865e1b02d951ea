"""Which groupwise 8-bit calls take the kernel of one launch (no workspace) and
which the split one, on 256 CUs: few steps of K (64, or 32 at group size 32) and
few rounds of 32 x 128 tiles stay in one launch."""

import pytest

from sparkq import _lib


@pytest.mark.parametrize("m,n,k,g,split", [
    (1, 64, 64, 64, False), (2048, 3072, 64, 64, False), (2048, 3200, 64, 64, True),
    (1, 32768, 192, 64, False), (128, 16384, 192, 64, False), (129, 16384, 128, 128, True),
    (256, 4096, 320, 64, False), (257, 4096, 320, 64, True), (1, 64, 384, 64, True),
    (1, 64, 32, 32, False), (512, 4096, 96, 32, False), (513, 4096, 96, 32, True),
    (256, 4096, 160, 32, False), (1, 64, 192, 32, True), (1, 2560, 4096, 32, True),
    (512, 3584, 2560, 64, True),
])
def test_route(m, n, k, g, split):
    assert (_lib.lib().sparkq_w8_affine_workspace_bytes(m, n, k, g) > 0) == split
