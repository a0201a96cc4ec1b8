"""Scratch buffers of the library calls: none is shared between two calls that are under way together."""
import threading

import pytest
import torch

from conftest import announce


def test_calls_have_scratch_of_their_own():
    _C = pytest.importorskip("bittorch_amd._C")
    a, b = (_C._workspace(4096, torch.device("cpu")) for _ in range(2))
    assert a.numel() >= 4096 and b.numel() >= 4096 and a.data_ptr() != b.data_ptr()
    assert _C._workspace(0, torch.device("cpu")) is None


def _work(seed):
    """Calls that make several launches around a scratch buffer: fp32 gradients, int8 products from float rows, fp32 rows."""
    from bittorch_amd import _C
    g = torch.Generator("cuda").manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    m, n, k = 2100 + 32 * seed, 256, 192
    packed, scale, _ = _C.ternary_quantize_pack(r(n, k) * 0.02, 0.05, True)
    x, dy = r(m, k), r(m, n)
    return lambda: (*_C.linear_grad_weight(dy, x, scale, True), _C.ternary_linear_tensor_core_forward(x, packed, scale, None, k),
                    _C.ternary_linear_packed_forward(x[:20], packed, scale, None, k))


@pytest.mark.gpu
def test_host_threads_on_one_stream():
    announce("scratch, threads")
    calls = [_work(s) for s in range(4)]
    want = [c() for c in calls]
    torch.cuda.synchronize()
    bad = []

    def loop(call, ref):
        for _ in range(50):
            got = call()
            bad.extend(i for i, (a, b) in enumerate(zip(got, ref)) if not torch.equal(a, b))

    threads = [threading.Thread(target=loop, args=cw) for cw in zip(calls, want)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad


@pytest.mark.gpu
def test_a_graph_keeps_its_scratch():
    """A later, larger call on the capture's stream takes nothing away from the recorded launches."""
    announce("scratch, graph")
    call, larger = _work(0), _work(40)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        want = call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        got = call()
    for _ in range(3):
        with torch.cuda.stream(stream):
            larger()
            fill = [torch.full((1 << 20,), float("nan"), device="cuda") for _ in range(8)]
        torch.cuda.synchronize()
        for t in got:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        del fill
