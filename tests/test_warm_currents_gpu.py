"""GPU: the warm-started forward where its predictions miss: constant and nearly constant currents
(trajectories of different phase never meet), ramps, steps, sub-threshold currents (the states meet
only when their last bits do) and NaN inputs.  The bits are the serial recurrence's, and the repair
stays within its budget: M/5 rounds and one serial sweep for M chunks."""
import numpy as np
import pytest
import torch

from oracle import lif_oracle as O
from tests._inputs import gpu, host, uniform

pytestmark = pytest.mark.gpu


def _current(kind, T, N):
    t = np.arange(T, dtype=np.float32)[:, None]
    x = {"constant": 0.15 + 0 * t, "threshold_below": 0.03 + 0 * t, "ramp": 0.05 + 0.2 * t / T,
         "steps": np.where(t % 700 < 350, 0.2, 0.0),
         "nearly_constant": 0.2 + 1e-3 * np.random.default_rng(2).standard_normal((T, N))}[kind]
    return np.ascontiguousarray(np.broadcast_to(x, (T, N)), dtype=np.float32)


KINDS = ["constant", "threshold_below", "ramp", "steps", "nearly_constant"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("T,N,C,W", [(4096, 128, 64, 256), (4096, 65, 32, 0), (2048, 3, 1024, 64)])
def test_repair_is_bounded(dev, kind, T, N, C, W):
    from lifscan import hip_lif as L
    I, u0 = _current(kind, T, N), uniform(N, 0.0, 1.0, 5)
    print(f"warm {kind} T={T} N={N} C={C} W={W}", flush=True)
    st = {}
    U, S = L.scan_forward_warm(gpu(I, dev), 0.93, 1.0, -0.1, gpu(u0, dev), C=C, W=W, stats=st)
    Uo, So = O.serial_forward(I, 0.93, 1.0, -0.1, u0)
    assert np.array_equal(host(U), Uo) and np.array_equal(host(S), So)
    assert st["repair_iters"] <= T // C // 5 + 1


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("T,N", [(12001, 70), (16384, 16)])
def test_layers_and_converged_scan(dev, kind, T, N):
    """The calls that choose warm-started chunks by themselves, a short last chunk among them."""
    from lifscan import hip_lif as L
    from lifscan.fit import lif_param
    I, u0 = _current(kind, T, N), uniform(N, 0.0, 1.0, 5)
    Uo, So = O.serial_forward(I, 0.93, 1.0, 0.0, u0)
    Ig, ug = gpu(I, dev), gpu(u0, dev)
    print(f"layers {kind} T={T} N={N}", flush=True)
    assert L.warm_any_plan(T, N, 0.93) is not None
    assert np.array_equal(host(L.lif_auto(Ig, ug, 0.93)), So)
    leaf = Ig.clone().requires_grad_(True)
    assert np.array_equal(host(L.lif_auto(leaf, ug, 0.93)), So)
    assert np.array_equal(host(lif_param(leaf, ug, 0.93, 1.0, 0.0)), So)
    C = 1 if T % 64 else 64
    U, S = L.scan_forward_v3(Ig, 0.93, 1.0, 0.0, ug, C=C, repair=T)
    assert np.array_equal(host(U), Uo) and np.array_equal(host(S), So)


@pytest.mark.parametrize("T,N,C,W", [(2048, 66, 64, 128), (2000, 3, 48, 96)])
def test_nan_and_infinite_inputs(dev, T, N, C, W):
    """A NaN stays in its neuron from its step on, an infinite input only where nothing spikes; the
    others are the serial sweep's bits."""
    from lifscan import hip_lif as L
    I, u0 = _current("steps", T, N), uniform(N, 0.0, 1.0, 5)
    I[301, 1], I[777, 0], I[900, 2] = np.nan, np.inf, -np.inf
    Ig, ug = gpu(I, dev), gpu(u0, dev)
    print(f"warm NaN T={T} N={N}", flush=True)
    U, S = L._warm_any(Ig, 0.93, 1.0, 0.0, ug, C, W)
    Us, Ss = L.serial_forward(Ig, 0.93, 1.0, 0.0, ug)
    assert torch.equal(S, Ss) and torch.equal(torch.nan_to_num(U, nan=7.0), torch.nan_to_num(Us, nan=7.0))
    assert bool(torch.isnan(U[301:, 1]).all()) and not bool(torch.isnan(U[:301]).any())


@pytest.mark.parametrize("kind", ["constant", "noise"])
def test_graph_replays(dev, kind):
    """A captured layer call on warm-started chunks, the serial sweep behind the rounds among them: every
    replay, with eager calls between, gives the eager spikes."""
    from lifscan import hip_lif as L
    T, N = 4096, 70
    assert L._auto_route(T, N, 0.93, False) == (256, 512)
    x = _current("constant", T, N) if kind == "constant" else None
    if x is None:
        x = (0.08 + 0.5 * np.random.default_rng(3).standard_normal((T, N))).astype(np.float32)
    u0 = uniform(N, 0.0, 1.0, 5)
    Ig, ug = gpu(x, dev), gpu(u0, dev)
    So = O.serial_forward(x, 0.93, 1.0, 0.0, u0)[1]
    with torch.no_grad():
        assert np.array_equal(host(L.lif_auto(Ig, ug, 0.93)), So)
        print(f"warm graph {kind}", flush=True)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            S = L.lif_auto(Ig, ug, 0.93)
        for _ in range(3):
            S.fill_(-1.0)
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(host(S), So)
            assert np.array_equal(host(L.lif_auto(Ig, ug, 0.93)), So)
