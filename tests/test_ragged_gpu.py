"""GPU: lengths that are no multiple of a kernel's tile, against the fp64 adjoint of the oracle."""
import numpy as np
import pytest
import torch

from oracle import lif_oracle as O
from tests._inputs import gpu, host, normal, uniform

pytestmark = pytest.mark.gpu


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


# one short segment; one step past a segment; a chunk and a wave past one; one step short of two
@pytest.mark.parametrize("T", [1, 17, 255, 257, 290, 511, 2081])
@pytest.mark.parametrize("N,detach,with_gu", [(1, True, False), (70, True, True), (130, False, True)])
def test_lookback_any_length(dev, T, N, detach, with_gu):
    """_lookback at every kind of last segment; the rows behind the inputs' last one are NaN, so a
    step past T that was read and used would show."""
    from lifscan import hip_lif as L
    I, GS = normal(T, N, 0.15, 0.4, T), normal(T, N, 0.0, 1.0, T + 1)
    GU = normal(T, N, 0.0, 0.3, T + 2) if with_gu else None
    u0 = uniform(N, 0.0, 1.0, 3)
    U, S = O.serial_forward(I, 0.95, 1.0, -0.1, u0)
    want = O.serial_backward(I, u0, U, S, GS, GU, 0.95, 1.0, -0.1, 4.0, detach, dtype=np.float64)
    pad = lambda a: torch.cat([gpu(a, dev), torch.full((300, N), float("nan"), device=dev)])[:T]
    args = [pad(I), gpu(u0, dev), pad(U), pad(S), pad(GS)]
    print(f"lookback any T={T} N={N}", flush=True)
    for C in (16, 32):
        Lam = L._lookback(*args, None if GU is None else pad(GU), 0.95, 1.0, -0.1, 4.0, detach, C=C)
        assert L.last_lookback_timeouts() == 0
        assert rel(host(Lam), want) < 1e-6  # fp32 recurrence: about 1e-7 of the fp64 one


@pytest.mark.parametrize("T,N", [(300, 65), (1001, 40), (2050, 130)])
def test_lookback_any_parameter_sums(dev, T, N):
    """lsh_lif_param_bwd and lsh_aff_bwd mode 4: Lam and the fp64 sums at ragged T."""
    from lifscan import fit
    from lifscan import hip_affine as AF
    beta, theta, u_r, gamma, delta = 0.93, 1.0, -0.1, 0.5, -0.25
    I, GS = normal(T, N, 0.08, 0.5, 7), normal(T, N, 0.0, 1.0, 8)
    u0 = uniform(N, 0.0, 1.0, 9)
    U, S = O.serial_forward(I, beta, theta, u_r, u0)
    Lam = O.serial_backward(I, u0, U, S, GS, None, beta, theta, u_r, 4.0, True, dtype=np.float64)
    want = O.param_grads(I, u0, U, S, GS, Lam, beta, theta, u_r, 4.0)
    print(f"param lookback any T={T} N={N}", flush=True)
    got, sums = fit._param_backward(*[gpu(a, dev) for a in (I, u0, U, S, GS)], beta, theta, u_r, 4.0,
                                    "lookback")
    assert rel(host(got), Lam) < 1e-6
    for k, g in enumerate((sums[0], -sums[1], beta * sums[2])):
        assert rel(g.item(), want[2 + k]) < 1e-4, k
    U, S = AF.aff_serial_forward(gpu(I, dev), beta, theta, gamma, delta, gpu(u0, dev))
    a = [gpu(I, dev), gpu(u0, dev), U, S, gpu(GS, dev), beta, theta, gamma, 4.0]
    l1, s1 = AF._aff_backward(*a, mode="lookback_any")
    l2, s2 = AF._aff_backward(*a, mode="serial")
    assert rel(host(l1), host(l2)) < 1e-6
    assert torch.allclose(s1, s2, rtol=1e-5, atol=1e-5 * float(s2.abs().max()))


def test_long_lengths_without_a_chunk_are_still_refused(dev):
    from lifscan import hip_affine as AF
    from lifscan import hip_lif as L
    z = lambda T, N=3: torch.zeros(T, N, device=dev)
    u0 = torch.zeros(3, device=dev)
    with pytest.raises(ValueError):
        L.scan_backward_tiled(z(1000), u0, z(1000), z(1000), z(1000), None, 0.9, 1.0, 0.0, C=64)
    with pytest.raises(ValueError):
        L.scan_backward_lookback(z(1000), u0, z(1000), z(1000), z(1000), None, 0.9, 1.0, 0.0)
    with pytest.raises(ValueError):
        AF._aff_backward(z(2049), u0, z(2049), z(2049), z(2049), 0.9, 1.0, 0.5, 4.0)


@pytest.mark.parametrize("T,N,C,W", [(1, 3, 256, 256), (257, 70, 256, 256), (4001, 65, 272, 0),
                                     (4095, 130, 256, 512), (4097, 64, 1024, 64)])
@pytest.mark.parametrize("beta,mu,sd", [(0.9, 0.12, 0.25), (0.99, 0.012, 0.08)])
def test_warm_forward_any_length(dev, T, N, C, W, beta, mu, sd):
    """The warm-started forward with a short last chunk is the serial recurrence bit for bit, also
    with warm-ups too short to predict anything (the repair's short chunk)."""
    from lifscan import hip_lif as L
    I, u0 = normal(T, N, mu, sd, T), uniform(N, 0.0, 1.0, 5)
    Uo, So = O.serial_forward(I, beta, 1.0, -0.1, u0)
    pad = torch.cat([gpu(I, dev), torch.full((300, N), float("nan"), device=dev)])[:T]
    print(f"warm any T={T} N={N} C={C} W={W}", flush=True)
    U, S = L._warm_any(pad, beta, 1.0, -0.1, gpu(u0, dev), C, W)
    assert np.array_equal(host(U), Uo) and np.array_equal(host(S), So)


def test_warm_any_plan_and_auto_layer(dev):
    """The layers' own forward at the bounds of the plan: the serial recurrence's spikes, and the
    adjoint of the look-back pass."""
    from lifscan import hip_lif as L
    assert L.warm_any_plan(2047, 64, 0.95) is None and L.warm_any_plan(2048, 64, 0.95) == (256, 512)
    assert L.warm_any_plan(60001, 64, 0.95) == (256, 512)
    assert L.warm_any_plan(4095, 4096, 0.95) is None and L.warm_any_plan(4096, 4096, 0.95) == (512, 512)
    assert L.warm_any_plan(10 ** 5, 4097, 0.9) is None and L.warm_any_plan(10 ** 5, 64, 1.0) is None
    T, N = 2501, 70
    I, GS = normal(T, N, 0.15, 0.4, 1), normal(T, N, 0.0, 1.0, 2)
    u0 = uniform(N, 0.0, 1.0, 3)
    Uo, So = O.serial_forward(I, 0.95, 1.0, 0.0, u0)
    want = O.serial_backward(I, u0, Uo, So, GS, None, 0.95, 1.0, 0.0, 4.0, True, dtype=np.float64)
    Ig, ug = gpu(I, dev).requires_grad_(True), gpu(u0, dev).requires_grad_(True)
    b = torch.tensor(0.95, device=dev, requires_grad=True)
    for beta in (0.95, b):
        S = L.lif_auto(Ig, ug, beta)
        dI, du0 = torch.autograd.grad(S, [Ig, ug], gpu(GS, dev), retain_graph=True)
        assert np.array_equal(host(S), So)
        assert rel(host(dI), want) < 1e-6 and rel(host(du0), 0.95 * want[0]) < 1e-6
    db, = torch.autograd.grad(S, [b], gpu(GS, dev))
    up = np.concatenate([u0[None], Uo[:-1]]).astype(np.float64)
    assert rel(db.item(), (want * up).sum()) < 1e-4


@pytest.mark.parametrize("N", [15, 16, 48, 49, 80, 129])
def test_row_alignment_store_policies(dev, N):
    """Both store policies (N % 16) of the serial sweeps, the recomputing pair, the replay and the
    ALIF layer: the oracle's bits and adjoints."""
    from lifscan import hip_lif as L
    from lifscan import triton_alif as A
    from oracle import alif_oracle as AO
    T = 160
    I, GS, u0 = normal(T, N, 0.15, 0.4, N), normal(T, N, 0.0, 1.0, N + 1), uniform(N, 0.0, 1.0, 3)
    Ig, Gg, ug = gpu(I, dev), gpu(GS, dev), gpu(u0, dev)
    Uo, So = O.serial_forward(I, 0.95, 1.0, 0.0, u0)
    want = O.serial_backward(I, u0, Uo, So, GS, None, 0.95, 1.0, 0.0, 4.0, True, dtype=np.float64)
    U, S = L.serial_forward(Ig, 0.95, 1.0, 0.0, ug)
    assert np.array_equal(host(U), Uo) and np.array_equal(host(S), So)
    S2, ST = L.scan_forward_exact_starts(Ig, 0.95, 1.0, 0.0, ug)
    assert np.array_equal(host(S2), So)
    lams = [L.serial_backward(Ig, ug, U, S, Gg, None, 0.95, 1.0, 0.0),
            L.scan_backward_fused_starts(Ig, ST, Gg, 0.95, 1.0, 0.0)[0],
            L.scan_backward_fused(Ig, ug, U, S, Gg, None, 0.95, 1.0, 0.0),
            L._lookback(Ig, ug, U, S, Gg, None, 0.95, 1.0, 0.0, 4.0, True)]
    for lam in lams:
        assert rel(host(lam), want) < 1e-6
    U3, S3 = L.scan_forward_mapscan(Ig, 0.95, 1.0, 0.0, ug, C=32, K=16, repair=10 ** 6)
    assert np.array_equal(host(U3), Uo) and np.array_equal(host(S3), So)
    w0 = np.zeros(N, np.float32)
    Ua, Wa, Sa = AO.serial_forward(I, 0.95, 0.995, 0.2, 1.0, 0.0, u0, w0)
    leaf = Ig.clone().requires_grad_(True)
    ps = [torch.tensor(v, device=dev, requires_grad=True) for v in (0.95, 0.995, 0.2, 1.0)]
    s, u, w = A.alif(leaf, ug, gpu(w0, dev), *ps)
    assert np.array_equal(host(s), Sa) and np.array_equal(host(u), Ua) and np.array_equal(host(w), Wa)
    dI, = torch.autograd.grad(s, [leaf], Gg)
    LV, _ = A.alif_backward(Ig, u, w, s, Gg, 0.95, 0.995, 0.2, 1.0, ug, gpu(w0, dev), mode="serial")
    assert rel(host(dI), host(LV)) < 1e-6


# the single pass, the look-back adjoint (T > 512, few neurons), the serial sweep forward (T > 768)
@pytest.mark.parametrize("T", [1, 31, 33, 257, 512, 513, 801])
@pytest.mark.parametrize("N", [1, 70, 129])
def test_layer_pair_any_length(dev, T, N):
    """The layers' forward and adjoint: the oracle's spikes and states bit for bit, the fp64 adjoint
    and parameter sums; rows behind the last one are NaN."""
    _layer_pair(dev, T, N)


def test_layer_pair_many_neurons(dev):
    _layer_pair(dev, 801, 16390)  # the single pass in both directions, a short last chunk


def _layer_pair(dev, T, N):
    from lifscan import _native as n
    from lifscan import hip_lif as L
    I, GS, u0 = normal(T, N, 0.15, 0.4, T), normal(T, N, 0.0, 1.0, T + 1), uniform(N, 0.0, 1.0, 3)
    U, S = O.serial_forward(I, 0.95, 1.0, -0.1, u0)
    want = O.serial_backward(I, u0, U, S, GS, None, 0.95, 1.0, -0.1, 4.0, True, dtype=np.float64)
    pad = lambda a: torch.cat([gpu(a, dev), torch.full((40, N), float("nan"), device=dev)])[:T]
    print(f"layer pair T={T} N={N}", flush=True)
    s, st = L._layer_forward(pad(I), 0.95, 1.0, -0.1, gpu(u0, dev))
    assert np.array_equal(host(s), S)
    assert np.array_equal(host(st), np.concatenate([u0[None], U[:-1]])[::32])
    s2, none = L._layer_forward(pad(I), 0.95, 1.0, -0.1, gpu(u0, dev), want_states=False)
    assert none is None and torch.equal(s2, s)
    lam, none = L._layer_backward(pad(I), st, pad(GS), 0.95, 1.0, -0.1)
    lam2, sums = L._layer_backward(pad(I), st, pad(GS), 0.95, 1.0, -0.1, 4.0, True)
    assert none is None and rel(host(lam), want) < 1e-6 and rel(host(lam2), want) < 1e-6
    if n.lib().lsh_lif_layer_bwd_workspace(T, N):  # the look-back adjoint: no wait gave up
        assert L.last_lookback_timeouts() == 0
    grads = O.param_grads(I, u0, U, S, GS, want, 0.95, 1.0, -0.1, 4.0)
    for k, g in enumerate((sums[0], -sums[1], 0.95 * sums[2])):
        assert abs(g.item() - grads[2 + k]) <= 1e-4 * abs(grads[2 + k]) + 1e-5, k
    assert L.starts_forward_timeouts(dev) == 0


@pytest.mark.parametrize("call", ["auto", "tuned", "param"])
@pytest.mark.parametrize("T,N", [(96, 40), (1002, 130), (1504, 5000)])
def test_layers_take_the_pair(dev, call, T, N):
    """lif_auto, lif_tuned (converged; T with a chunk) and lif_param: spikes, dI, du0 and dbeta."""
    from lifscan import hip_lif as L
    from lifscan.fit import lif_param
    if call == "tuned" and T == 1002:
        with pytest.raises(ValueError):  # no chunk for T: refused, as ever
            L.lif_tuned(torch.zeros(T, N, device=dev), torch.zeros(N, device=dev), repair=10 ** 6)
        return
    I, GS, u0 = normal(T, N, 0.15, 0.4, 1), normal(T, N, 0.0, 1.0, 2), uniform(N, 0.0, 1.0, 3)
    Uo, So = O.serial_forward(I, 0.95, 1.0, 0.0, u0)
    want = O.serial_backward(I, u0, Uo, So, GS, None, 0.95, 1.0, 0.0, 4.0, True, dtype=np.float64)
    Ig, ug = gpu(I, dev).requires_grad_(True), gpu(u0, dev).requires_grad_(True)
    b = torch.tensor(0.95, device=dev, requires_grad=True)
    f = {"auto": lambda x: L.lif_auto(Ig, ug, x), "tuned": lambda x: L.lif_tuned(Ig, ug, x, repair=10 ** 6),
         "param": lambda x: lif_param(Ig, ug, x, 1.0, 0.0)}[call]
    for beta in (0.95, b):
        S = f(beta)
        grads = torch.autograd.grad(S, [Ig, ug] + ([b] if beta is b else []), gpu(GS, dev))
        assert np.array_equal(host(S), So)
        assert rel(host(grads[0]), want) < 1e-6 and rel(host(grads[1]), 0.95 * want[0]) < 1e-6
    up = np.concatenate([u0[None], Uo[:-1]]).astype(np.float64)
    assert abs(grads[2].item() - (want * up).sum()) <= 1e-4 * abs((want * up).sum()) + 1e-4
    with torch.no_grad():
        assert np.array_equal(host(f(0.95)), So)


def test_scan_arguments_are_still_refused(dev):
    """A map capacity or repair budget that the scans refuse is refused whichever forward runs."""
    from lifscan import hip_lif as L
    from lifscan.fit import lif_param
    I, u0 = torch.zeros(16384, 8, device=dev), torch.zeros(8, device=dev)
    assert L.warm_any_plan(16384, 8, 0.9) is not None
    for kw in ({"K": 0}, {"K": 65}, {"repair": -1}):
        with pytest.raises(ValueError):
            L.lif_auto(I, u0, 0.9, **kw)
    for K in (0, 65):
        with pytest.raises(ValueError):
            lif_param(I, u0, 0.9, 1.0, 0.0, K=K)
    with pytest.raises(ValueError):  # the layer pair
        L.lif_tuned(I[:96], u0, 0.9, K=0, repair=10 ** 6)
    with pytest.raises(ValueError):  # warm-started chunks of a T without a power-of-two chunk
        L.scan_forward_v3(I[:2064], 0.9, 1.0, 0.0, u0, C=16, K=0, repair=10 ** 6)
    assert L.lif_auto(I, u0, 0.9, K=64).shape == I.shape  # what was taken still is
    assert L.lif_tuned(I[:96], u0, 0.9, K=32, repair=10 ** 6).shape == (96, 8)


@pytest.mark.parametrize("call", ["auto", "tuned", "param"])
@pytest.mark.parametrize("T,N,C", [(1024, 1024, 0), (4096, 70, 256)])
def test_few_neuron_layers_run_from_cpp(dev, call, T, N, C):
    """The few-neuron layers, the warm-started chunks among them, run as C++ functions with a look-back
    adjoint behind the forward, and without gradients as spikes alone."""
    from lifscan import hip_lif as L
    from lifscan.fit import lif_param
    assert L.layer_warm_plan(T, N, 0.9) == ((C, 256) if C else None)
    I, GS, u0 = normal(T, N, 0.12, 0.25, 1), normal(T, N, 0.0, 1.0, 2), uniform(N, 0.0, 1.0, 3)
    Uo, So = O.serial_forward(I, 0.9, 1.0, 0.0, u0)
    want = O.serial_backward(I, u0, Uo, So, GS, None, 0.9, 1.0, 0.0, 4.0, True, dtype=np.float64)
    Ig, ug = gpu(I, dev).requires_grad_(True), gpu(u0, dev).requires_grad_(True)
    f = {"auto": lambda: L.lif_auto(Ig, ug, 0.9), "tuned": lambda: L.lif_tuned(Ig, ug, 0.9, repair=10 ** 6),
         "param": lambda: lif_param(Ig, ug, 0.9, 1.0, 0.0)}[call]
    print(f"layers {call} T={T} N={N}", flush=True)
    S = f()
    assert "LIFLayer" in S.grad_fn.name()
    dI, du0 = torch.autograd.grad(S, [Ig, ug], gpu(GS, dev))
    assert np.array_equal(host(S), So)
    assert rel(host(dI), want) < 1e-6 and rel(host(du0), 0.9 * want[0]) < 1e-6
    with torch.no_grad():
        assert np.array_equal(host(f()), So)


@pytest.mark.parametrize("N", [8191, 8193, 16401])
def test_store_policies_of_many_neurons(dev, N):
    """Rows that are no multiple of 64 bytes on both sides of the kernels' least numbers of neurons for
    plain stores."""
    from lifscan import hip_lif as L
    from lifscan import triton_affine as AF
    from oracle import affine_oracle as AO
    test_row_alignment_store_policies(dev, N)
    T = 64
    I, GS, u0 = normal(T, N, 0.15, 0.4, N), normal(T, N, 0.0, 1.0, N + 1), uniform(N, 0.0, 1.0, 3)
    Ig, Gg, ug = gpu(I, dev), gpu(GS, dev), gpu(u0, dev)
    Uo, So = O.serial_forward(I, 0.95, 1.0, 0.0, u0)
    want = O.serial_backward(I, u0, Uo, So, GS, None, 0.95, 1.0, 0.0, 4.0, True, dtype=np.float64)
    U, S = L.scan_forward_exact(Ig, 0.95, 1.0, 0.0, ug, maps=False)
    assert np.array_equal(host(U), Uo) and np.array_equal(host(S), So)
    S, ST = L._layer_forward(Ig[:63], 0.95, 1.0, 0.0, ug)
    assert np.array_equal(host(S), So[:63])
    assert np.array_equal(host(ST), np.stack([u0, Uo[31]]))
    lam, sums = L._layer_backward(Ig, L._layer_forward(Ig, 0.95, 1.0, 0.0, ug)[1], Gg, 0.95, 1.0, 0.0, 4.0, True)
    assert rel(host(lam), want) < 1e-6
    Ua, Sa = AO.serial_forward(I, 0.95, 1.0, 0.5, -0.25, u0)
    U, S = AF.aff_serial_forward(Ig, 0.95, 1.0, 0.5, -0.25, ug)
    assert np.array_equal(host(U), Ua) and np.array_equal(host(S), Sa)
