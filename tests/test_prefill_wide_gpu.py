"""The prefill kernel of 32 query columns per wave and its slices of the cache: at the edges of its
column units (32 columns a wave, 128 a workgroup), tiles (32 positions) and slice counts, for several
group sizes, against the oracle (bars as in test_prefill_gpu.py), with strided gate and output rows;
the fp8 cache against the bf16 cache bit for bit; sliced against unsliced; under graph capture."""
import pytest
import torch

import oracle as O
from attn_cases import BF, D, attn_close, gen

pytestmark = pytest.mark.gpu
DEV = "cuda"

CASES = [
    # (Hq, Hkv, T, pos, max_len)
    (6, 1, 5, 0, 5),           # 30 columns: less than one wave
    (24, 4, 43, 0, 64),        # 258 columns: two in the third unit
    (16, 2, 16, 0, 16),        # exactly one unit
    (16, 2, 17, 495, 512),     # rows below and above 512 positions (one and two terms of P)
    (1, 1, 129, 3, 132),       # one row a column, two units
    (64, 1, 3, 40, 43),        # a row over two waves
    (12, 4, 70, 1000, 1100),   # group size 3: rows straddle waves
    (24, 4, 100, 3000, 3100),  # slices of the cache
    (24, 4, 30, 9000, 9030),   # many slices of one or two tiles
    (8, 2, 40, 2000, 1500),    # rows past the end of the cache attend the whole cache
]


def inputs(hq, hkv, T, max_len, seed=0):
    g = gen(1000 * hq + T + seed)
    kc, vc = (torch.randn(hkv, max_len, D, generator=g).to(BF) for _ in range(2))
    q = torch.randn(T, hq * D, generator=g).to(BF)
    qg = torch.randn(T, hq * 2 * D + 64, generator=g).to(BF)[:, : hq * 2 * D]  # strided rows
    return q, kc, vc, qg


def dev_rows(x):
    """x on the GPU with its row stride."""
    return torch.empty(x.shape[0], x.stride(0), dtype=x.dtype, device=DEV)[:, : x.shape[1]].copy_(x)


def run(op, q, kc, vc, pos, qg, *scales):
    T, hq = q.shape[0], q.shape[1] // D
    out = torch.full((T, hq * D + 8), float("nan"), dtype=BF, device=DEV)[:, : hq * D]
    op(q.to(DEV), kc.to(DEV), vc.to(DEV), torch.tensor([pos], dtype=torch.int32, device=DEV),
       dev_rows(qg), out, *scales)
    torch.cuda.synchronize()
    return out.cpu()


@pytest.mark.parametrize("hq,hkv,T,pos,max_len", CASES)
def test_wide_prefill(native, hq, hkv, T, pos, max_len):
    q, kc, vc, qg = inputs(hq, hkv, T, max_len)
    out = run(native.attn_prefill, q, kc, vc, pos, qg)
    ok, mx, mean = attn_close(out, O.attn_prefill(q, kc, vc, pos, qg, hq))
    assert ok, (mx, mean)
    k8, v8 = kc.to(torch.float8_e4m3fn), vc.to(torch.float8_e4m3fn)
    a = run(native.attn_prefill_fp8, q, k8, v8, pos, qg, 1.0, 1.0)
    b = run(native.attn_prefill, q, k8.to(BF), v8.to(BF), pos, qg)
    assert torch.equal(a, b)


@pytest.mark.parametrize("hq,hkv,T,pos", [(24, 4, 100, 3000), (16, 2, 9, 12000), (6, 1, 700, 2600)])
def test_slices_match_unsliced(native, capi, hq, hkv, T, pos):
    """The op slices the cache; the C entry point without a workspace does not. Both round the same
    fp32 result to bf16 and differ by the order of sums alone (fp32, and P's bf16 rounding against
    another running maximum): far inside the oracle's bar."""
    max_len = pos + T
    assert capi.load().qe_attn_prefill_ws_size(T, hq, hkv, max_len) > 0
    q, kc, vc, qg = inputs(hq, hkv, T, max_len, 1)
    a = run(native.attn_prefill, q, kc, vc, pos, qg)
    qd, kd, vd, gd = q.to(DEV), kc.to(DEV), vc.to(DEV), dev_rows(qg)
    p = torch.tensor([pos], dtype=torch.int32, device=DEV)
    b = torch.empty(T, hq * D, dtype=BF, device=DEV)
    assert capi.prefill(qd, kd, vd, p, gd, gd.stride(0), b, hq * D, T, hq, hkv, max_len) == 0
    ok, mx, mean = attn_close(a, b.cpu())
    assert ok and mean <= 2e-4, (mx, mean)


def test_captured_prefill_equals_unsliced(native, capi):
    """Under capture the op takes no workspace: replays, with the position changed in place and eager
    calls between them, equal the unsliced entry point bit for bit."""
    hq, hkv, T, max_len = 24, 4, 60, 4096
    q, kc, vc, qg = inputs(hq, hkv, T, max_len, 2)
    qd, kd, vd, gd = q.to(DEV), kc.to(DEV), vc.to(DEV), dev_rows(qg)
    p = torch.tensor([3000], dtype=torch.int32, device=DEV)
    out, ref, eager = (torch.empty(T, hq * D, dtype=BF, device=DEV) for _ in range(3))
    native.attn_prefill(qd, kd, vd, p, gd, out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        native.attn_prefill(qd, kd, vd, p, gd, out)
    for pos in (3000, 0, 4000, 1234):
        p.fill_(pos)
        out.fill_(float("nan"))
        graph.replay()
        native.attn_prefill(qd, kd, vd, p, gd, eager)
        assert capi.prefill(qd, kd, vd, p, gd, gd.stride(0), ref, hq * D, T, hq, hkv, max_len) == 0
        torch.cuda.synchronize()
        assert torch.equal(out, ref), pos
        ok, mx, mean = attn_close(eager.cpu(), ref.cpu())
        assert ok, (pos, mx, mean)


def test_negative_scale(capi):
    """The C entry point takes any scale; a negative one equals the positive one on negated q."""
    hq, hkv, T, pos = 6, 1, 50, 300
    q, kc, vc, qg = inputs(hq, hkv, T, pos + T, 3)
    kd, vd, gd = kc.to(DEV), vc.to(DEV), dev_rows(qg)
    p = torch.tensor([pos], dtype=torch.int32, device=DEV)
    a, b = (torch.empty(T, hq * D, dtype=BF, device=DEV) for _ in range(2))
    args = (gd, gd.stride(0))
    assert capi.prefill(q.to(DEV), kd, vd, p, *args, a, hq * D, T, hq, hkv, pos + T, -1.0 / 16) == 0
    assert capi.prefill(-q.to(DEV), kd, vd, p, *args, b, hq * D, T, hq, hkv, pos + T, 1.0 / 16) == 0
    torch.cuda.synchronize()
    assert torch.isfinite(a.float()).all() and torch.equal(a, b)


@pytest.mark.parametrize("pos", [0, 3000])  # one pass over the cache, and slices
def test_every_gate(native, pos):
    """All 65,536 bf16 gates: with K = 0 and V = 1 the attention is exactly 1, and the output is the
    gate's sigmoid. The decode op evaluates it by the library's exponential and a division; the prefill
    has the same bits (-87.5 .. -88.5 give subnormal values)."""
    hq, hkv, T = 16, 2, 16
    gates = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(BF).view(T, hq, 1, D)
    qg = torch.cat([torch.zeros_like(gates), gates], 2).reshape(T, -1).to(DEV)
    kc = torch.zeros(hkv, pos + T, D, dtype=BF, device=DEV)
    q, vc = torch.zeros(T, hq * D, dtype=BF, device=DEV), torch.ones_like(kc)
    out, ref = torch.empty_like(q), torch.empty_like(q)
    p = torch.tensor([pos], dtype=torch.int32, device=DEV)
    native.attn_prefill(q, kc, vc, p, qg, out)
    po, pml = torch.empty(8, hq, 16, D, device=DEV), torch.empty(8, hq, 16, 2, device=DEV)
    for t in (0, 8):
        native.attn_decode(q[t:t + 8], kc, vc, p + t, qg[t:t + 8], po, pml, ref[t:t + 8])
    nan = ref.isnan()
    assert torch.equal(out.isnan(), nan)
    assert torch.equal(out.view(torch.int16)[~nan], ref.view(torch.int16)[~nan])
    assert ((ref > 0) & (ref.float() < 1.17e-38)).any()


@pytest.mark.parametrize("sliced", [False, True])
def test_least_v_scale(native, capi, sliced):
    """O / L is rounded before V's scale multiplies it: the scale's least values (1.2e-38) give the bits
    of a scale 2^100 times as large, times 2^-100, although scale / L would be subnormal."""
    hq, hkv, T, pos = 16, 2, 16, 12000
    g = gen(9)
    q = torch.randn(T, hq * D, generator=g).to(BF).to(DEV)
    kc = torch.randn(hkv, pos + T, D, generator=g).to(torch.float8_e4m3fn).to(DEV)
    vc = (1 + 400 * torch.rand(hkv, pos + T, D, generator=g)).to(torch.float8_e4m3fn).to(DEV)
    qg = torch.full((T, hq * 2 * D), 60.0, dtype=BF, device=DEV)  # gates of 1
    p = torch.tensor([pos], dtype=torch.int32, device=DEV)
    scale = torch.tensor(1.2e-38, dtype=torch.float32).item()
    outs = []
    for vs in (scale, scale * 2.0 ** 100):
        out = torch.empty_like(q)
        if sliced:
            native.attn_prefill_fp8(q, kc, vc, p, qg, out, 1.0, vs)
        else:
            assert capi.prefill_fp8(q, kc, vc, p, qg, qg.stride(0), out, hq * D, T, hq, hkv, pos + T,
                                    1.0, vs) == 0
        outs.append(out.double())
    assert outs[0].min() > 1.18e-38  # normal values
    assert torch.equal(outs[0], outs[1] * 2.0 ** -100)


def test_infinite_v(native):
    """An infinity in V comes out as an infinity where the rows attend it with weight (one bf16 term of
    P: beyond 512 positions), as from a division; dims without one are not touched."""
    q, kc, vc, qg = inputs(6, 1, 40, 1040, 4)
    vc[0, 3, 5], vc[0, 4, 9] = float("inf"), float("-inf")
    out = run(native.attn_prefill, q, kc, vc, 1000, torch.zeros_like(qg)).float().view(40, 6, D)
    assert (out[:, :, 5] == float("inf")).all() and (out[:, :, 9] == float("-inf")).all()
    out[:, :, 5] = out[:, :, 9] = 0
    assert torch.isfinite(out).all()


@pytest.mark.parametrize("hq,hkv", [(24, 4), (8, 2), (4, 4)])
def test_rows_of_two_term_blocks(native, hq, hkv):
    """P keeps two bf16 terms for every row of a 16-row block that begins below 512 attended positions,
    whatever rows a wave holds: rows 400 .. 415 of a chunk at position 103 (504 .. 519 positions) are
    within fp32 sums of the exact attention, so that nearly every output is its bf16 rounding. (One term
    is 2e-3 off, more than half of bf16's spacing for about two values in five.)"""
    T, pos = 416, 103
    q, kc, vc, qg = inputs(hq, hkv, T, pos + T, 5)
    out = run(native.attn_prefill, q, kc, vc, pos, torch.full_like(qg, 60.0))  # gates of 1
    rows, grp = range(400, 416), hq // hkv
    K, V, Q = kc.double(), vc.double(), q.view(T, hq, D).double()
    same = []
    for r in rows:
        L = pos + r + 1
        for h in range(hq):
            p = torch.softmax(K[h // grp, :L] @ Q[r, h] / 16, 0)
            same.append(out.view(T, hq, D)[r, h] == (p @ V[h // grp, :L]).to(BF))
    share = torch.stack(same).float().mean(1).view(len(rows), hq).mean(1)
    assert share.min() > 0.99, share


@pytest.mark.parametrize("hq,hkv,T,pos", [(4, 2, 70, 0), (4, 2, 129, 40), (2, 2, 33, 0), (10, 2, 27, 5),
                                          (14, 2, 19, 0)])
def test_group_sizes(native, hq, hkv, T, pos):
    """Rows and heads of a lane's columns for group sizes that divide, straddle and exceed its step of two
    columns, with rows that end inside a wave."""
    q, kc, vc, qg = inputs(hq, hkv, T, pos + T, 6)
    out = run(native.attn_prefill, q, kc, vc, pos, qg)
    ok, mx, mean = attn_close(out, O.attn_prefill(q, kc, vc, pos, qg, hq))
    assert ok, (mx, mean)
