"""GPU: the layers' C++ autograd functions (lifscan/_ops.cpp) against the Python autograd functions
over the same kernels: S, dL/dI and dL/du0 are the same bits; the parameter gradients sum the same
fp64 partials in another order and are rounded to fp32 at other places, so they may differ by
3 * 2^-24 of themselves plus the reordering of at most T * N terms, 2^-53 * T * N * sum |term|."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _data(T, N, dev, seed=7):
    g = torch.Generator().manual_seed(seed)
    I = (0.12 + 0.25 * torch.randn(T, N, generator=g)).to(dev)
    return I, torch.randn(T, N, generator=g).to(dev), (0.3 * torch.rand(N, generator=g)).to(dev)


def _both(fns, T, N, params, dev, u0_grad=True, wide_grad=True):
    I, gS, u0 = _data(T, N, dev)
    outs = []
    for fn, cpp in zip(fns, (True, False)):
        Ig = I.clone().requires_grad_(True)
        ug = u0.clone().requires_grad_(u0_grad)
        ps = [torch.tensor(p, device=dev, requires_grad=r) for p, r in params]
        S = fn(Ig, ug, *ps)
        # each side ran as what it is compared as
        assert ("LIFLayer" in S.grad_fn.name() or "AffLayer" in S.grad_fn.name()) == cpp, S.grad_fn.name()
        if wide_grad:
            S.backward(gS)
        else:
            S.sum().backward()
        outs.append((S.detach(), Ig.grad, ug.grad, [p.grad for p in ps]))
    (S1, dI1, du1, g1), (S2, dI2, du2, g2) = outs
    assert torch.equal(S1, S2) and torch.equal(dI1, dI2)
    assert (du1 is None and du2 is None) or torch.equal(du1, du2)
    terms = float(dI2.double().abs().sum()) * (1.0 + float(I.abs().max()) * 10)
    for a, b in zip(g1, g2):
        assert (a is None) == (b is None)
        if a is not None:
            assert a.shape == b.shape == ()
            assert abs(float(a) - float(b)) <= 3 * 2.0 ** -24 * abs(float(b)) + 2.0 ** -53 * T * N * terms


@pytest.mark.parametrize("T,N", [(1, 1), (33, 65), (1001, 77), (513, 4096), (769, 130), (256, 16391)])
@pytest.mark.parametrize("grads", [(True,), (False,)])
def test_auto_layer(dev, T, N, grads):
    from lifscan import hip_lif as L
    assert L._cpp_u0(*(_data(T, N, dev)[k] for k in (0, 2))) is not None
    print(f"auto T={T} N={N}", flush=True)
    fwd, bwd = L.auto_modes(N, T)
    fwd, bwd = L._auto_fwd(fwd, N, T), L._auto_bwd(bwd, N, T)
    _both((lambda I, u0, b: L.lif_auto(I, u0, b),
           lambda I, u0, b: L.LIFAuto.apply(I, u0, b, 1.0, 0.0, 4.0, 16, 0, fwd, bwd)),
          T, N, [(0.95, grads[0])], dev, u0_grad=grads[0], wide_grad=grads[0])


@pytest.mark.parametrize("T,N", [(1, 3), (700, 130), (4099, 64), (8192, 200), (31, 20000)])
@pytest.mark.parametrize("which", [(True, True, True), (False, True, False)])
def test_param_layer(dev, T, N, which):
    from lifscan import fit as F
    from lifscan import hip_lif as L
    print(f"param T={T} N={N}", flush=True)
    fwd, bwd = L.auto_modes(N, T)
    fwd, bwd = L._auto_fwd(fwd, N, T), L._auto_bwd(bwd, N, T)
    _both((lambda I, u0, *p: F.lif_param(I, u0, *p),
           lambda I, u0, *p: F.LIFParamFn.apply(I, u0, *p, 4.0, fwd, bwd, 16, True)),
          T, N, list(zip((0.9, 1.0, 0.05), which)), dev)


@pytest.mark.parametrize("T,N,mode", [(128, 1, "scan"), (2048, 200, "scan"), (1152, 333, "scan"),
                                      (100, 65, "serial"), (256, 16391, "serial")])
@pytest.mark.parametrize("soft", [False, True])
def test_affine_and_soft_layer(dev, T, N, mode, soft):
    from lifscan import fit as F
    from lifscan import hip_affine as AF
    print(f"soft={soft} T={T} N={N} {mode}", flush=True)
    if soft:
        fns = (lambda I, u0, b: F.lif_soft_scan(I, u0, b, mode=mode),
               lambda I, u0, b: F.LIFSoftScanFn.apply(I, u0, b, 1.0, 4.0, mode, 128, 32))
        params = [(0.9, True)]
    else:
        fns = (lambda I, u0, *p: AF.lif_affine(I, u0, *p, mode=mode),
               lambda I, u0, *p: AF.LIFAffineFn.apply(I, u0, *p, 1.0, 4.0, mode, 128, 32))
        params = [(0.9, True), (0.5, False), (-0.25, True)]
    _both(fns, T, N, params, dev)


def test_calls_that_stay_with_the_python_functions(dev):
    from lifscan import hip_lif as L
    I, _, u0 = _data(64, 32, dev)
    theta = torch.tensor(1.0, device=dev, requires_grad=True)
    assert L._cpp_u0(I, u0, theta) is None  # keeps its (empty) gradient edge
    assert L._cpp_u0(I.double(), u0) is None and L._cpp_u0(I.cpu(), u0) is None
    assert L._cpp_u0(I, u0.double().requires_grad_(True)) is None
    assert L.lif_auto(I, u0, 0.95, theta).requires_grad
    with torch.autograd.forward_ad.dual_level():
        assert L._cpp_u0(I, u0) is None


def test_parameters_under_a_function_transform(dev):
    """Parameters that a transform has wrapped have no storage of their own to copy; the scans read
    their values as those of any other constant."""
    from lifscan import hip_lif as L
    I, _, u0 = _data(64, 32, dev)
    want = L.serial_forward(I, 0.95, 1.0, 0.05, u0)
    got = []

    def loss(p):
        got.append(L._f32s(p[0], p[1], p[2]))
        return p.sum()

    torch.func.grad(loss)(torch.tensor([0.95, 1.0, 0.05], device=dev))
    assert got[0] == tuple(torch.tensor([0.95, 1.0, 0.05]).tolist())
    assert all(map(torch.equal, L.serial_forward(I, *got[0], u0), want))


@pytest.mark.parametrize("P,cols,N", [(0, 3, 5), (1, 1, 1), (511, 3, 512), (513, 1, 513), (70001, 3, 64)])
def test_layer_grads_kernel(dev, P, cols, N):
    from lifscan import _native as n
    g = torch.Generator().manual_seed(3)
    parts = torch.randn(max(P, 1), cols, generator=g, dtype=torch.float64).to(dev)
    lam = torch.randn(N, generator=g).to(dev)
    sums = torch.empty(cols, device=dev)
    du0 = torch.empty(N, device=dev)
    n.check(n.lib().lsh_layer_grads(n.ptr(parts), P, cols, 1.0, -1.0, 0.95, n.ptr(sums), n.ptr(lam), N,
                                    0.95, n.ptr(du0), n.stream_of(lam)), "lsh_layer_grads")
    s = torch.tensor([1.0, -1.0, 0.95], dtype=torch.float64, device=dev)[:cols]
    p = parts[:P]
    tol = 2.0 ** -24 * (s * p.sum(0)).abs() + 2.0 ** -52 * P * p.abs().sum(0)
    assert bool(((sums.double() - s * p.sum(0)).abs() <= tol).all())
    assert torch.equal(du0, 0.95 * lam)


@pytest.mark.parametrize("T", [96, 4096, 4128])  # the pair, and plans with and without a power-of-two chunk
@pytest.mark.parametrize("call", ["tuned", "tuned_scan", "auto"])
def test_device_beta_is_read_once(dev, monkeypatch, T, call):
    """A beta on the device is read by one synchronizing copy a call, also where plans depend on it."""
    from lifscan import hip_lif as L
    I, gS, u0 = _data(T, 70, dev)
    I.requires_grad_(True)
    beta = torch.tensor(0.9, device=dev, requires_grad=True)
    fn = {"tuned": lambda: L.lif_tuned(I, u0, beta, repair=10 ** 6), "tuned_scan": lambda: L.lif_tuned(I, u0, beta),
          "auto": lambda: L.lif_auto(I, u0, beta)}[call]
    want = fn().detach()
    reads = []
    item = torch.Tensor.item
    monkeypatch.setattr(torch.Tensor, "item", lambda self: (reads.append(1), item(self))[1])
    S = fn()
    assert len(reads) == 1 and torch.equal(S, want)
    dI, db = torch.autograd.grad(S, [I, beta], gS)
    assert len(reads) == 1 and dI.shape == I.shape and db.shape == ()
