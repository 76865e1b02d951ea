"""Which causal prompts at head dim 256 the affine prefill runs in halves of
tiles: the workspace query is nonzero for those and zero for whole tiles (from
one tile of 128 rows per CU on; 256 CUs)."""

import pytest

from sparkq import _lib


def _halves(b, hq, hkv, length, n, d=256, causal=1):
    return _lib.lib().sparkq_int8kv_sdpa_prefill_affine_workspace_bytes(
        b, hq, hkv, length, n, d, causal) > 0


@pytest.mark.parametrize("b,hq,hkv,length,n", [
    (1, 16, 4, 2048, 2048), (1, 16, 4, 2048, 3072), (1, 16, 4, 2304, 2304), (1, 8, 2, 4096, 4096),
    (1, 16, 2, 2048, 2048), (1, 16, 16, 2056, 2056),
    (1, 16, 4, 3104, 3104), (1, 16, 4, 4064, 4064),  # not dealt as whole tiles
])
def test_halves(b, hq, hkv, length, n):
    assert _halves(b, hq, hkv, length, n)


@pytest.mark.parametrize("b,hq,hkv,length,n,causal", [
    (1, 16, 4, 2048, 3073, 1), (1, 16, 4, 2048, 16384, 1), (1, 16, 4, 2048, 2048, 0),
    (2, 16, 4, 1024, 1024, 1), (4, 16, 4, 512, 512, 1), (8, 16, 4, 256, 256, 1),
    (3, 16, 4, 700, 700, 1), (1, 16, 4, 2560, 2560, 1), (1, 16, 4, 3072, 3072, 1),
    (1, 20, 5, 2688, 2688, 1), (1, 24, 6, 2112, 2112, 1), (2, 16, 4, 1424, 1424, 1),
    (1, 8, 2, 8000, 8000, 1), (1, 16, 4, 4096, 4096, 1), (1, 64, 8, 512, 512, 1),
])
def test_whole_tiles(b, hq, hkv, length, n, causal):
    assert not _halves(b, hq, hkv, length, n, causal=causal)


@pytest.mark.parametrize("d", [64, 128])
def test_other_head_dims_run_whole(d):
    assert not _halves(1, 16, 4, 2048, 2048, d)
