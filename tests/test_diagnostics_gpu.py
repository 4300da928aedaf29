"""GPU: what the accessors of the most recent run describe: the run itself, whichever route a layer's
forward or adjoint took."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_last_scan_run_after_warm_chunks_of_any_length(dev):
    from lifscan import hip_lif as L
    u0 = torch.zeros(3, device=dev)
    L.scan_forward_mapscan(torch.zeros(128, 3, device=dev), 0.9, 1.0, 0.0, u0, C=64, K=16)
    T = 2064
    L.scan_forward_v3(torch.zeros(T, 3, device=dev), 0.9, 1.0, 0.0, u0, C=16, repair=T)
    run = L.last_scan_run()
    assert run.warm and (run.C, run.W) == L.warm_any_plan(T, 3, 0.9)


def _adjoints():
    from lifscan import fit as F
    from lifscan import hip_affine as AF
    from lifscan import hip_lif as L
    return {"pair": (600, lambda I, u0, b: L.lif_auto(I, u0, b)),
            "pair_python": (600, lambda I, u0, b: L.LIFAuto.apply(I, u0, b, 1.0, 0.0, 4.0, 16, 0, "serial",
                                                                  "scan")),
            "warm": (4099, lambda I, u0, b: F.lif_param(I, u0, b, 1.0, 0.0)),
            "warm_python": (4099, lambda I, u0, b: F.LIFParamFn.apply(I, u0, b, 1.0, 0.0, 4.0, "auto",
                                                                      "lookback", 16, True)),
            "affine": (256, lambda I, u0, b: AF.lif_affine(I, u0, b, 0.5, -0.25)),
            "affine_python": (256, lambda I, u0, b: AF.LIFAffineFn.apply(I, u0, b, 0.5, -0.25, 1.0, 4.0,
                                                                         "scan", 128, 32))}


@pytest.mark.parametrize("name", ["pair", "pair_python", "warm", "warm_python", "affine", "affine_python"])
def test_last_lookback_is_the_layers(dev, name):
    from lifscan import hip_lif as L
    T, fn = _adjoints()[name]
    other = torch.zeros(256, dtype=torch.uint8, device=dev)
    L._note_lookback(other)
    assert L.last_lookback_timeouts() == 0
    I = (0.12 + 0.25 * torch.randn(T, 70, generator=torch.Generator().manual_seed(1))).to(dev)
    b = torch.tensor(0.9, device=dev, requires_grad=True)
    print(f"look-back {name}", flush=True)
    fn(I.requires_grad_(True), torch.zeros(70, device=dev), b).sum().backward()
    assert L._last_lookback().data_ptr() != other.data_ptr()
    assert L.last_lookback_timeouts() == 0


def test_check_waits_reads_the_lookback(dev, monkeypatch):
    """With LIFSCAN_CHECK_WAITS a count other than 0 in a look-back's header raises."""
    from lifscan import hip_lif as L
    monkeypatch.setattr(L, "CHECK_WAITS", True)
    L._note_lookback(torch.zeros(256, dtype=torch.uint8, device=dev))
    with pytest.raises(RuntimeError):
        L._note_lookback(torch.ones(256, dtype=torch.uint8, device=dev))
    monkeypatch.setattr(L, "CHECK_WAITS", False)
    L._note_lookback(torch.zeros(256, dtype=torch.uint8, device=dev))
