"""Every row count of a Gated DeltaNet step at the start of a sequence, where each conv thread's
window mixes rows of the call, ring slots and positions before the sequence: row t of an n-row call
equals one-row calls bit for bit (outputs, committed state, staged rows, ring)."""
import pytest
import torch

from test_gdn_gpu import gpu_layer, make_rows, weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("start", [0, 1, 2, 3, 15])
@pytest.mark.parametrize("n", range(1, 9))
def test_rows_at_the_start(native, n, start):
    hk, hv = 2, 6
    W = weights(hk, hv, seed=n)
    many, ones = gpu_layer(native, hk, hv, W), gpu_layer(native, hk, hv, W)
    before = make_rows(hk, hv, 16, seed=5)
    for t in range(start):
        assert torch.equal(many.run(before[t:t + 1], 1), ones.run(before[t:t + 1], 1))
    rows = make_rows(hk, hv, n, seed=start)
    out = many.run(rows, n)
    for t in range(n):
        assert torch.equal(out[t], ones.run(rows[t:t + 1], 1)[0]), t
    last = make_rows(hk, hv, 1, seed=77)
    assert torch.equal(many.run(last, 1), ones.run(last, 1))
    assert torch.equal(many.S, ones.S) and torch.equal(many.ring, ones.ring)
    for a, b in zip(many.st, ones.st):
        assert torch.equal(a[0], b[0])
