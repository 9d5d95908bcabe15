"""Slices of one, two and three tiles: the shortened merges give the general merge's bits.

A slice of one tile writes wave 0's accumulators directly (1 column tile), and one of at most two
tiles leaves out the empty subsets' zero terms. Row t of an n-row call (kernels with 1, 2, 3 and 4
column tiles) equals the 1-row call at pos + t bit for bit, and the call meets the oracle's bar.
"""
import pytest
import torch

from attn_cases import attn_close, decode_case
from test_attn_gpu import gpu_decode, oracle_decode

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiles", [1, 2, 3])
@pytest.mark.parametrize("hq,hkv,n", [(24, 4, 1), (24, 4, 2), (24, 4, 5), (24, 4, 8), (16, 2, 8)])
def test_few_tile_slices(native, tiles, hq, hkv, n):
    ns = 6
    pos = 32 * tiles * ns - n - 5  # every slice holds `tiles` tiles, the last one a ragged tile
    case = decode_case(seed=pos + n, hq=hq, hkv=hkv, pos=pos, n=n, max_len=pos + n + 3)
    out = gpu_decode(native, case, ns)
    ok, mx, mean = attn_close(out, oracle_decode(case))
    assert ok, (mx, mean)
    for t in range(n):
        one = gpu_decode(native, case, ns, pos=pos + t, rows=slice(t, t + 1))
        assert torch.equal(one[0], out[t]), t
        few = gpu_decode(native, case, 1, pos=pos + t, rows=slice(t, t + 1))  # the general merge
        ok, mx, mean = attn_close(few, out[t:t + 1])
        assert ok, (t, mx, mean)
