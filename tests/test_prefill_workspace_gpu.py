"""The workspace of the chunked prefill: where it comes from and what it may not disturb."""
import threading

import pytest
import torch

from attn_cases import BF, D

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
