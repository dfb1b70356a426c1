"""Forwards that use the library's second stream, captured into a HIP graph: two calls in one capture, replayed several
times on changing inputs with eager calls of the same paths between the replays; every replay equals the eager result."""
import pytest
import torch

from scan_inputs import scan_inputs

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import slotkern_hip as KH


# a chunk pipeline, batch groups, and the register chain
@pytest.mark.parametrize("B,T,N,D", [(2, 600, 70, 64), (300, 100, 130, 128), (300, 40, 130, 128)])
def test_captured_forwards_equal_eager_ones(B, T, N, D):
    print("capture", B, T, N, D, flush=True)
    draws = [[x.cuda() for x in scan_inputs(B, T, 1, D, 60 + i, dtype=torch.bfloat16)] for i in range(3)]
    temp = torch.tensor(16.0, device="cuda")
    buf = [x.clone() for x in draws[0]]

    def calls(x):
        k, q, v, g, fr = x
        kw = dict(G=8, q=q, occ_bin=True)
        with torch.no_grad():
            kb, vb, st = KH.kv_scan_stream(k, v, g, fr, N, temp, **kw)
            mem = KH.kv_scan_mem(k, v, g, fr, N, temp, hard=True, detach_addr=True, **kw)
        return [kb, vb, *st, *mem]

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        calls(buf)                                       # outside the capture first: streams, events, code
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = calls(buf)
    for i in (0, 1, 2, 1, 0):
        for b, x in zip(buf, draws[i]):
            b.copy_(x)
        graph.replay()
        got = [o.clone() for o in out]
        eager = calls(draws[i])                          # beside the graph, on the same second stream
        for a, b in zip(got, eager):
            assert torch.equal(a, b)
        torch.cuda.synchronize()
