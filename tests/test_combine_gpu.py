"""The decode combine alone, on partials made by the partials kernel: slice counts around its batches
of 64, and rows of gates and outputs with and without 8-byte alignment.

Expected: the fp64 log-sum-exp merge of the same fp32 partials. Three bf16 roundings (O / L, the
sigmoid, their product) of relative 2^-8 at most each separate the two; 1e-5 covers the fp32 sums of
up to 260 slices where O cancels."""
import pytest
import torch

from attn_cases import BF, D, decode_case

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rows(x, shift):
    """x on the GPU, `shift` elements past an allocation's start, with a row stride of width + shift."""
    n, wd = x.shape
    flat = torch.zeros(shift + n * (wd + shift), dtype=x.dtype, device=DEV)
    v = flat[shift:].view(n, wd + shift)[:, :wd]
    return v.copy_(x)


@pytest.mark.parametrize("ns,pos", [(63, None), (64, None), (65, None), (128, None), (129, None),
                                    (192, None), (193, None), (260, None), (200, 100), (130, 2080)])
def test_combine_batches(native, ns, pos):
    n, hq, hkv = 2, 4, 1
    pos = 32 * ns - n - 3 if pos is None else pos  # else fewer slices than slots
    case = decode_case(seed=ns, hq=hq, hkv=hkv, pos=pos, n=n, max_len=pos + n + 5)
    q, kc, vc = (t.to(DEV) for t in (case.q, case.kc, case.vc))
    p = torch.tensor([pos], dtype=torch.int32, device=DEV)
    po = torch.full((n, hq, ns, D), float("nan"), device=DEV)   # slots without a slice stay NaN
    pml = torch.full((n, hq, ns, 2), float("nan"), device=DEV)
    outs = []
    for shift in (0, 1, 4):
        qg, out = rows(case.qg, shift), rows(torch.zeros(n, hq * D, dtype=BF), shift)
        if shift == 0:
            native.attn_decode_partials(q, kc, vc, p, qg, po, pml, out)
        native.attn_decode_combine(q, kc, vc, p, qg, po, pml, out)
        outs.append(out.cpu())
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    for t in range(n):
        L = pos + t + 1
        S = -(-L // (-(-(-(-L // ns)) // 32) * 32))  # slices of ceil(L / ns) positions, whole tiles
        m, l = pml[t, :, :S].double().unbind(-1)
        w = torch.exp2(m - m.amax(-1, keepdim=True))
        o = (po[t, :, :S].double() * w[..., None]).sum(1) / (l * w).sum(-1)[:, None]
        gate = case.qg[t].view(hq, 2, D)[:, 1].to(DEV).double()
        want = (o * torch.sigmoid(gate)).reshape(-1).cpu()
        err = (outs[0][t].double() - want).abs()
        assert (err <= 3.1 * 2 ** -8 * want.abs() + 1e-5).all(), (t, err.max().item())
