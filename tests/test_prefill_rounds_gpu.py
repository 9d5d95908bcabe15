"""Both prefill kernels at the call sizes the small tests do not reach: the balanced kernel (GQA 6) with
whole, ragged and part-empty rounds of workgroups, and the kernel of 32 columns per wave with whole
rounds of units, a remainder of them (in slices and unsplit), and more slices than tiles. Each on the
bf16 and the fp8 cache.

Expected: the attention in fp64 (on the GPU, one head at a time) with the op's three bf16 roundings; bars
as in test_prefill_gpu.py. Which kernel a shape runs is asserted from the dispatch rule and the device's
compute units, so that a change of the rule cannot empty a test."""
import math

import pytest
import torch

import qengine_amd as qa
from attn_cases import BF, D, attn_close

pytestmark = pytest.mark.gpu
DEV = "cuda"
F8 = torch.float8_e4m3fn


def make(hq, hkv, T, pos, max_len, kv8, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed + T)

    def randn(*shape):
        return torch.randn(shape, generator=g, device=DEV).to(BF)

    q, qg = randn(T, hq * D), randn(T, hq * 2 * D)
    kc, vc = randn(hkv, max_len, D), randn(hkv, max_len, D)
    end = min(pos + T, max_len)
    kc[:, end:] = vc[:, end:] = float("nan")  # nothing past the attended rows may matter
    if kv8:
        kc, vc = kc.to(F8), vc.to(F8)
    return q, kc, vc, torch.tensor([pos], dtype=torch.int32, device=DEV), qg


def exact(q, kc, vc, pos, qg, ks=1.0, vs=1.0):
    """The op in fp64, rounded to bf16 where it rounds."""
    T, hq, hkv, max_len = q.shape[0], q.shape[1] // D, kc.shape[0], kc.shape[1]
    L = min(pos + T, max_len)
    ends = (torch.arange(T, device=DEV) + pos + 1).clamp(max=max_len)
    hidden = torch.arange(L, device=DEV)[None] >= ends[:, None]
    out = torch.empty(T, hq, D, dtype=BF, device=DEV)
    for h in range(hq):
        K, V = (c[h // (hq // hkv), :L].to(torch.float32).double() for c in (kc, vc))
        s = q.view(T, hq, D)[:, h].double() @ (K * (ks / 16)).t().contiguous()
        o = (torch.softmax(s.masked_fill_(hidden, -math.inf), -1) @ (V * vs)).to(BF)
        gate = qg.view(T, hq, 2, D)[:, h, 1].float().sigmoid().to(BF)
        out[:, h] = o * gate
    return out.view(T, hq * D)


def call(capi, q, kc, vc, p, qg, ws=None, scales=(1.0, 1.0)):
    """One call through the C entry points: on a workspace, or without."""
    T, hq, hkv, max_len = q.shape[0], q.shape[1] // D, kc.shape[0], kc.shape[1]
    out = torch.full((T, hq * D), float("nan"), dtype=BF, device=DEV)
    kv8 = kc.dtype == F8
    args = (q, kc, vc, p, qg, qg.stride(0), out, hq * D, T, hq, hkv, max_len, *(scales if kv8 else ()))
    if ws is None:
        assert (capi.prefill_fp8 if kv8 else capi.prefill)(*args) == 0
    else:
        assert (capi.prefill_fp8_ws if kv8 else capi.prefill_ws)(*args, ws, ws.numel()) == 0
    torch.cuda.synchronize()
    return out


def check(out, ref):
    ok, mx, mean = attn_close(out.cpu(), ref.cpu())
    assert ok, (mx, mean)


# (Hq, Hkv, T, pos, max_len): balanced on 256 compute units, without a workspace
BALANCED = [
    (24, 4, 1953, 0, 6000),     # 123 blocks: the last one ragged, an odd number of pairs
    (24, 4, 1999, 700, 6000),   # 125 blocks: a half pair, no KV head per XCD
    (24, 4, 2047, 1500, 3000),  # rows past the end of the cache; KV heads on XCDs of their own
    (24, 4, 1500, 300, 5500),   # 188 workgroups, an odd number per KV head
    (12, 2, 3500, 0, 9000),
    (48, 8, 900, 100, 9000),    # one XCD per KV head
    (6, 1, 8000, 0, 9000),
    (24, 4, 4096, 0, 20096),    # two rounds; alone, the bf16 cache's fastest kernel is the other one
    (24, 4, 6144, 0, 22144),    # three rounds
]


@pytest.mark.parametrize("kv8", [False, True])
@pytest.mark.parametrize("hq,hkv,T,pos,max_len", BALANCED)
def test_balanced(native, capi, hq, hkv, T, pos, max_len, kv8):
    if qa.compute_units() == 256:
        assert capi.load().qe_attn_prefill_balanced(T, hq, hkv, max_len, 0)
    scales = (2.0, 0.5) if kv8 else (1.0, 1.0)
    q, kc, vc, p, qg = make(hq, hkv, T, pos, max_len, kv8)
    check(call(capi, q, kc, vc, p, qg, scales=scales), exact(q, kc, vc, pos, qg, *scales))
    if kv8:  # scales of 1: the bf16 cache's bits
        a = call(capi, q, kc, vc, p, qg)
        b = call(capi, q, kc.to(BF), vc.to(BF), p, qg)
        assert torch.equal(a, b)


@pytest.mark.parametrize("kv8", [False, True])
def test_balanced_two_term_rows(native, capi, kv8):
    """Rows attending fewer than 512 positions keep P in two bf16 terms: with gates of 1 nearly every
    value is the exact attention's bf16 rounding (one term: about 3 in 5)."""
    hq, hkv, T, pos, max_len = 24, 4, 1999, 7, 6000
    if qa.compute_units() == 256:
        assert capi.load().qe_attn_prefill_balanced(T, hq, hkv, max_len, 0)
    q, kc, vc, p, qg = make(hq, hkv, T, pos, max_len, kv8, seed=3)
    qg.fill_(60.0)
    out, ref = call(capi, q, kc, vc, p, qg), exact(q, kc, vc, pos, qg)
    assert (out[:496] == ref[:496]).float().mean(1).min() > 0.97  # 6,144 values a row
    assert (out[:496] == ref[:496]).float().mean() > 0.99


# (Hq, Hkv, T, pos), U units of 128 columns on W workgroups of a KV head (256 compute units)
ROUNDS = [
    (32, 8, 1100, 3000),  # U = 35, W = 32: one round, 3 units left
    (24, 4, 1400, 1000),  # U = 66, W = 64, GQA 6
    (32, 8, 1024, 100),   # U = W
    (16, 2, 4200, 0),     # U = 263, W = 128: two rounds, 7 units left
    (8, 1, 40, 250),      # U = 3, W = 256: more slices than tiles
    (4, 1, 9000, 2000),   # U = 282, W = 256
]


@pytest.mark.parametrize("kv8", [False, True])
@pytest.mark.parametrize("hq,hkv,T,pos", ROUNDS)
def test_rounds_of_units(native, capi, hq, hkv, T, pos, kv8):
    max_len = pos + T
    if qa.compute_units() == 256:
        U, W = -(-T * (hq // hkv) // 128), 256 // hkv
        assert U >= W or T == 40
        need = capi.prefill_ws_need(T, hq, hkv, max_len)
        assert (need > 0) == (U % W != 0)
        assert not capi.load().qe_attn_prefill_balanced(T, hq, hkv, max_len, 1)
    scales = (2.0, 0.5) if kv8 else (1.0, 1.0)
    q, kc, vc, p, qg = make(hq, hkv, T, pos, max_len, kv8)
    ref = exact(q, kc, vc, pos, qg, *scales)
    ws = qa.alloc_prefill_ws(T, hq, hkv, max_len).fill_(0xFF)
    check(call(capi, q, kc, vc, p, qg, ws, scales), ref)
    check(call(capi, q, kc, vc, p, qg, scales=scales), ref)
