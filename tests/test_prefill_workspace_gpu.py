"""The workspace of the chunked prefill: where it comes from and what it may not disturb."""
import threading

import pytest
import torch

from attn_cases import BF, D, attn_close

pytestmark = pytest.mark.gpu
DEV = "cuda"


def case(hq, hkv, T, pos, max_len=None, seed=0):
    """q, K and V cache, position, gate rows and an output of one call, on the GPU."""
    max_len = pos + T if max_len is None else max_len
    g = torch.Generator(device=DEV).manual_seed(seed)

    def randn(*shape):
        return torch.randn(shape, generator=g, device=DEV).to(BF)

    q, qg = randn(T, hq * D), randn(T, hq * 2 * D)
    kc, vc = randn(hkv, max_len, D), randn(hkv, max_len, D)
    p = torch.tensor([pos], dtype=torch.int32, device=DEV)
    return q, kc, vc, p, qg, torch.full((T, hq * D), float("nan"), dtype=BF, device=DEV)


def test_allocates_beside_another_threads_capture(native):
    """An eager chunk whose workspace is not in torch's pool, while another thread captures a graph in
    the global mode (which forbids device allocations to every thread in the default mode): the chunk
    is computed, and the capture ends and replays as if alone."""
    *args, out = case(24, 4, 64, 4000)
    ref = torch.empty_like(out)
    native.attn_prefill(*args, ref)
    x = torch.zeros(1000, device=DEV)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    raised, grown = [], []

    def other():
        before = torch.cuda.memory_reserved()
        try:
            with torch.cuda.stream(side):
                native.attn_prefill(*args, out)
        except RuntimeError as e:
            raised.append(str(e))
        grown.append(torch.cuda.memory_reserved() - before)

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, capture_error_mode="global"):
        x.add_(1)
        thread = threading.Thread(target=other)
        thread.start()
        thread.join()
        x.add_(1)
    assert not raised and grown[0] > 0, (raised, grown)  # it did allocate
    for n in (1, 2, 3):
        graph.replay()
        torch.cuda.synchronize()
        assert (x == 2 * n).all()
    assert torch.equal(out, ref)


SHAPES = [
    # (Hq, Hkv, T, pos, max_len)
    (16, 2, 9, 12000, 12100),    # one unit a KV head in many slices
    (24, 4, 301, 5000, 5400),    # 15 units, 4 slices each
    (32, 8, 1100, 3000, 4100),   # a whole round of units ahead of a remainder in slices (256 CUs)
    (24, 4, 1400, 2000, 3400),   # the same, GQA 6
    (24, 4, 40, 100, 9000),      # short prefix in a long cache: fewer slices than the workspace holds
    (8, 2, 40, 5000, 3000),      # rows past the end of the cache
]


@pytest.mark.parametrize("kv8", [False, True])
@pytest.mark.parametrize("hq,hkv,T,pos,max_len", SHAPES)
def test_caller_workspace(native, capi, hq, hkv, T, pos, max_len, kv8):
    """The C entry points on a workspace of exactly qe_attn_prefill_ws_need() bytes, full of NaN and
    between guards: the op's bits, guards untouched. One byte less runs unsplit (the bits of the entry
    point without a workspace); a misaligned one is rejected."""
    q, kc, vc, p, qg, out = case(hq, hkv, T, pos, max_len)
    need = capi.prefill_ws_need(T, hq, hkv, max_len)
    assert need > 0 and need % 16 == 0
    if kv8:
        kc, vc = kc.to(torch.float8_e4m3fn), vc.to(torch.float8_e4m3fn)
    scales = (0.5, 2.0) if kv8 else ()
    guard = 4096
    buf = torch.full((guard + need + guard,), 0xFF, dtype=torch.uint8, device=DEV)  # fp32 NaN
    ws = buf.data_ptr() + guard
    args = (q, kc, vc, p, qg, qg.stride(0))
    rest = (hq * D, T, hq, hkv, max_len)
    run_ws = capi.prefill_fp8_ws if kv8 else capi.prefill_ws
    plain = capi.prefill_fp8 if kv8 else capi.prefill
    op = native.attn_prefill_fp8 if kv8 else native.attn_prefill
    ref, unsplit = torch.empty_like(out), torch.empty_like(out)
    op(q, kc, vc, p, qg, ref, *scales)
    assert plain(*args, unsplit, *rest, *scales) == 0
    assert run_ws(*args, out, *rest, *scales, ws, need) == 0
    torch.cuda.synchronize()
    assert torch.isfinite(out.float()).all() and torch.equal(out, ref)
    assert (buf[:guard] == 0xFF).all() and (buf[guard + need:] == 0xFF).all()
    assert run_ws(*args, out.fill_(float("nan")), *rest, *scales, ws, need - 1) == 0
    assert torch.equal(out, unsplit)
    assert run_ws(*args, out.fill_(float("nan")), *rest, *scales, None, 0) == 0
    assert torch.equal(out, unsplit)
    assert run_ws(*args, out, *rest, *scales, ws + 8, need) == capi.HIP_ERROR_INVALID_VALUE
    ok, mx, mean = attn_close(ref.cpu(), unsplit.cpu())
    assert ok, (mx, mean)


def test_op_allocates_what_it_needs(native, capi):
    """An eager chunk takes the bytes that its slices need from torch's allocator, and holds none of
    them once it has returned."""
    *args, out = case(16, 2, 9, 8000)
    native.attn_prefill(*args, out)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    native.attn_prefill(*args, out)
    need = capi.prefill_ws_need(9, 16, 2, 8009)
    assert need <= torch.cuda.max_memory_allocated() - before <= need + (2 << 20)
    assert torch.cuda.memory_allocated() == before


@pytest.mark.parametrize("kv8", [False, True])
def test_captured_on_a_caller_workspace_equals_eager(native, kv8):
    """On a caller's workspace a captured chunk splits the cache as the eager op does: every replay, the
    position changed in place and eager calls between them, has the eager op's bits. The call allocates
    nothing."""
    import qengine_amd as qa
    hq, hkv, T, max_len = 24, 4, 60, 4096
    q, kc, vc, p, qg, out = case(hq, hkv, T, 3000, max_len)
    if kv8:
        kc, vc = kc.to(torch.float8_e4m3fn), vc.to(torch.float8_e4m3fn)
    scales = (0.5, 2.0) if kv8 else ()
    op = native.attn_prefill_fp8 if kv8 else native.attn_prefill
    op_ws = native.attn_prefill_fp8_ws if kv8 else native.attn_prefill_ws
    ws = qa.alloc_prefill_ws(T, hq, hkv, max_len)
    assert ws.numel() > 0
    eager = torch.empty_like(out)
    op_ws(q, kc, vc, p, qg, out, *scales, ws)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    op_ws(q, kc, vc, p, qg, out, *scales, ws)
    assert torch.cuda.max_memory_allocated() == before
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        op_ws(q, kc, vc, p, qg, out, *scales, ws)
    for pos in (3000, 0, 4000, 1234):
        p.fill_(pos)
        out.fill_(float("nan"))
        ws.fill_(0xFF)
        graph.replay()
        op(q, kc, vc, p, qg, eager, *scales)
        torch.cuda.synchronize()
        assert torch.equal(out, eager), pos


def test_workspace_op_rejects(native):
    """A workspace that is misaligned, strided or elsewhere is refused; an empty one runs unsplit."""
    q, kc, vc, p, qg, out = case(24, 4, 60, 3000)
    ws = torch.empty(1 << 26, dtype=torch.uint8, device=DEV)
    for bad, why in ((ws[8:], "aligned"), (ws[::2], "contiguous"), (ws.cpu(), "device")):
        with pytest.raises(RuntimeError, match=why):
            native.attn_prefill_ws(q, kc, vc, p, qg, out, bad)
    native.attn_prefill_ws(q, kc, vc, p, qg, out, ws[:0])
    ref = torch.empty_like(out)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):  # attn_prefill takes no workspace under capture
        native.attn_prefill(q, kc, vc, p, qg, ref)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, ref)
