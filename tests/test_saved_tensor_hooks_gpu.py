"""GPU: the layers under saved-tensor hooks.  What a hook hands back in a tensor of other strides gives
the same gradients; a tensor that is no longer the float32 one on the GPU that was saved is refused
before a kernel gets its address."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _layers():
    from lifscan import fit as F
    from lifscan import hip_affine as AF
    from lifscan import hip_lif as L
    return {"pair": (96, lambda I, u0, b: L.lif_auto(I, u0, b)),
            "warm": (4099, lambda I, u0, b: F.lif_param(I, u0, b, 1.0, 0.0)),
            "tuned": (96, lambda I, u0, b: L.lif_tuned(I, u0, b, repair=10 ** 6)),
            "affine": (256, lambda I, u0, b: AF.lif_affine(I, u0, b, 0.5, -0.25)),
            "soft": (256, lambda I, u0, b: F.lif_soft_scan(I, u0, b)),
            "python": (97, lambda I, u0, b: L.LIFAuto.apply(I, u0, b, 1.0, 0.0, 4.0, 16, 0, "serial", "serial"))}


def _run(fn, T, dev, pack, unpack):
    N = 70
    g = torch.Generator().manual_seed(T)
    I = (0.12 + 0.25 * torch.randn(T, N, generator=g)).to(dev).requires_grad_(True)
    gS = torch.randn(T, N, generator=g).to(dev)
    u0 = (0.3 * torch.rand(N, generator=g)).to(dev).requires_grad_(True)
    b = torch.tensor(0.9, device=dev, requires_grad=True)
    with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
        S = fn(I, u0, b)
    return torch.autograd.grad(S, [I, u0, b], gS)


@pytest.mark.parametrize("name", ["pair", "warm", "tuned", "affine", "soft", "python"])
def test_hooks(dev, name):
    T, fn = _layers()[name]
    print(f"hooks {name}", flush=True)
    same = lambda t: t
    want = _run(fn, T, dev, same, same)
    strided = lambda t: t.t().contiguous().t() if t.dim() == 2 else torch.stack([t, t], -1)[..., 0]
    for a, b in zip(_run(fn, T, dev, same, strided), want):
        assert torch.equal(a, b)
    for other in (lambda t: t.cpu(), lambda t: t.half(), lambda t: t[:-1] if t.dim() else t.cpu()):
        with pytest.raises(ValueError):
            _run(fn, T, dev, same, other)
