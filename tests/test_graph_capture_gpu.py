"""The two-level map scan captured in a HIP graph (through torch.cuda.CUDAGraph) and replayed:
its launches take torch's current stream, clear the workspace header with a kernel (no memset
node) and read nothing back when no statistics are asked for, so a captured call can be
replayed.  Every replay, with eager calls and synchronizations between them, gives the eager
result bit for bit: with few neurons (one-wave-per-neuron carry) and with many (staged carry).
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [128, 4096])
def test_map_scan_graph_replays(dev, N):
    from lifscan import hip_lif as L
    T, C, K, beta = 16384, 128, 16, 0.99
    g = torch.Generator().manual_seed(63)
    I = (0.15 + 0.4 * torch.randn(T, N, generator=g)).to(dev)
    u0 = torch.zeros(N, device=dev)
    print(f"map scan graph replays N={N}", flush=True)
    U0, S0 = L.scan_forward_mapscan(I, beta, 1.0, 0.0, u0, C=C, K=K, repair=0)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        L.scan_forward_mapscan(I, beta, 1.0, 0.0, u0, C=C, K=K, repair=0)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        U, S = L.scan_forward_mapscan(I, beta, 1.0, 0.0, u0, C=C, K=K, repair=0)
    for _ in range(3):
        U.fill_(-1.0)
        S.fill_(-1.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(U, U0) and torch.equal(S, S0)
        U1, S1 = L.scan_forward_mapscan(I, beta, 1.0, 0.0, u0, C=C, K=K, repair=0)
        torch.cuda.synchronize()
        assert torch.equal(U1, U0) and torch.equal(S1, S0)


def test_first_layer_call_in_a_capture(dev):
    """A layer whose first call is captured: the graph clears a counter header of its own, and the
    process's header, which starts_forward_timeouts reads, is not one that only a replay clears."""
    from lifscan import hip_lif as L
    g = torch.Generator().manual_seed(3)
    I = (0.15 + 0.4 * torch.randn(100, 70, generator=g)).to(dev)
    u0 = torch.zeros(70, device=dev)
    with torch.no_grad():
        want = L.lif_auto(I, u0, 0.95)
        kept = dict(L._WAIT_HEADERS)
        L._WAIT_HEADERS.clear()
        try:
            print("layer graph", flush=True)
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                S = L.lif_auto(I, u0, 0.95)
            assert not L._WAIT_HEADERS
            for _ in range(3):
                S.fill_(-1.0)
                graph.replay()
                torch.cuda.synchronize()
                assert torch.equal(S, want)
                assert torch.equal(L.lif_auto(I, u0, 0.95), want) and L.starts_forward_timeouts(dev) == 0
        finally:
            L._WAIT_HEADERS.update(kept)
