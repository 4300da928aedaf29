"""The work that programs give this framework, as cases that can be timed and checked.

A case names a path through the public entry points and its sizes.  listed() holds one case or
two of every path, draw() more of the same ranges, prepare() makes what a program has in hand
before the call, run() is one pass, exact() the same outputs from plain torch.

  infer      spikes of a layer without gradients (lif_auto under no_grad)
  layer      a layer's training step: spikes, dI, du0 (lif_auto, any number of steps)
  tuned      the same through lif_tuned with repair, the headline layer
  long       few neurons, long sequences, beta near 1: exact forward and scan adjoint
  mapscan    scan_forward_v3 as called by default (chunk maps, no repair)
  threelevel scan_forward_v4 as called by default
  fit        neuron-parameter fitting: lif_param with gradients for beta, theta, u_r
  alif       an adaptive-threshold layer's training step with its four parameter gradients
  alifbox    the adaptive layer's box scan from a warm-up prediction
  affine     affine-reset layer with gradients for beta, gamma, delta
  soft       soft-reset layer with the gradient for beta
  net        a training step's gradients of the two-layer spiking classifier

A trajectory is defined in fp32: two roundings a step, v = fl(fl(beta*u) + x), and the spikes are
the sign of a comparison, so a 64-bit forward would be another spike train after the first tie.
exact() therefore steps the forward in fp32 and takes everything behind it, surrogate, adjoints and
parameter sums, in 64 bits.
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "hard-resets-compose_amd"))

from lifscan import fit as F  # noqa: E402
from lifscan import triton_affine as AF  # noqa: E402
from lifscan import triton_alif as A  # noqa: E402
from lifscan import triton_lif as L  # noqa: E402
from lifscan.shdnet import Net  # noqa: E402

DEVICE = "cuda"
# mean and standard deviation of the currents that go with a decay (the repository's benchmark)
CURRENTS = {0.9: (0.12, 0.25), 0.93: (0.08, 0.5), 0.95: (0.15, 0.4), 0.99: (0.012, 0.08)}
ALPHA = 4.0
RHO, Q = 0.995, 0.2          # adaptation decay and jump of the adaptive layers
GAMMA, DELTA = 0.5, -0.25    # affine reset
U_R_FIT = -0.1               # reset value of the fitted neurons
CONVERGE = 10 ** 6           # repair budget of a converged call


# ----------------------------------------------------------------------------- the cases
def listed():
    return [
        # one 256-neuron layer on a 100-step window of one recording: launches and latency count
        {"name": "infer_small", "path": "infer", "T": 100, "N": 256, "beta": 0.95},
        # a batch of 50 x 256 neurons over 1000 steps: T is a multiple of no power of two over 8
        {"name": "layer_ragged", "path": "layer", "T": 1000, "N": 12800, "beta": 0.95},
        # the headline benchmark's layer, 256 x 256 neurons: bandwidth counts
        {"name": "tuned_wide", "path": "tuned", "T": 4096, "N": 65536, "beta": 0.9, "K": 8},
        # a long recording through a small layer: parallel over time or not at all
        {"name": "long_narrow", "path": "long", "T": 262144, "N": 1024, "beta": 0.99, "C": 64},
        # the two-level scan with the default chunk and capacity
        {"name": "mapscan_mid", "path": "mapscan", "T": 4096, "N": 8192, "beta": 0.9, "C": 64, "K": 16},
        # the three-level scan with its defaults on a long sequence
        {"name": "threelevel_long", "path": "threelevel", "T": 65536, "N": 1024, "beta": 0.99, "C": 64,
         "G": 16},
        # one step of fitting 64 neurons to 50 s of recording at 1 kHz
        {"name": "fit_recording", "path": "fit", "T": 50000, "N": 64, "beta": 0.93},
        # the benchmark's adaptive layer
        {"name": "alif_layer", "path": "alif", "T": 4096, "N": 16384, "beta": 0.95},
        # the adaptive forward as a scan, a layer of 1024 neurons
        {"name": "alifbox_mid", "path": "alifbox", "T": 16384, "N": 1024, "beta": 0.95, "C": 128},
        # the test suite's affine-reset shape
        {"name": "affine_narrow", "path": "affine", "T": 8192, "N": 200, "beta": 0.9},
        # the test suite's soft-reset shape
        {"name": "soft_narrow", "path": "soft", "T": 8192, "N": 333, "beta": 0.95},
        # the classifier of the benchmark, batch 64
        {"name": "net_step", "path": "net", "T": 1024, "N": 64, "beta": 0.95, "H": 256},
    ]


def _spread(rng, lo, hi):
    """A whole number between lo and hi, spread over the logarithm, odd ones as likely as even."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _sizes(rng, t, n, most):
    """T and N in the ranges t and n with T*N <= most."""
    T = _spread(rng, *t)
    return T, _spread(rng, n[0], max(n[0], min(n[1], most // T)))


def draw(rng):
    path = rng.choice(["infer", "layer", "layer", "tuned", "long", "mapscan", "threelevel", "fit", "alif",
                       "alifbox", "affine", "soft", "net"])
    beta = rng.choice([0.9, 0.95, 0.99])
    if path == "infer":
        T, N = _sizes(rng, (16, 4096), (64, 65536), 2 ** 26)
        return {"path": path, "T": T, "N": N, "beta": beta}
    if path == "layer":
        T, N = _sizes(rng, (64, 8192), (64, 65536), 2 ** 27)
        return {"path": path, "T": T, "N": N, "beta": beta}
    if path == "tuned":
        T, N = _sizes(rng, (4, 128), (64, 65536), 2 ** 22)
        return {"path": path, "T": 32 * T, "N": N, "beta": beta, "K": rng.choice([8, 16])}
    if path == "long":
        T, N = _sizes(rng, (256, 4096), (16, 4096), 2 ** 22)
        return {"path": path, "T": 64 * T, "N": N, "beta": rng.choice([0.9, 0.99]), "C": 64}
    if path == "mapscan":
        C = rng.choice([32, 64, 128])
        T, N = _sizes(rng, (8, 8192 // C), (64, 16384), 2 ** 25 // C)
        return {"path": path, "T": C * T, "N": N, "beta": beta, "C": C, "K": rng.choice([8, 16])}
    if path == "threelevel":
        C, G = rng.choice([(64, 16), (128, 8)])
        T, N = _sizes(rng, (8, 128), (64, 2048), 2 ** 16)
        return {"path": path, "T": C * G * T, "N": N, "beta": rng.choice([0.9, 0.99]), "C": C, "G": G}
    if path == "fit":
        T, N = _sizes(rng, (1000, 60000), (1, 512), 2 ** 23)
        return {"path": path, "T": T, "N": N, "beta": rng.choice([0.9, 0.93])}
    if path == "alif":
        T, N = _sizes(rng, (4, 512), (64, 32768), 2 ** 22)  # the adjoint takes multiples of 16
        return {"path": path, "T": 16 * T, "N": N, "beta": rng.choice([0.9, 0.95])}
    if path == "alifbox":
        C = rng.choice([128, 256])
        T, N = _sizes(rng, (8, 128), (16, 4096), 2 ** 24 // C)
        return {"path": path, "T": C * T, "N": N, "beta": rng.choice([0.9, 0.95]), "C": C}
    if path in ("affine", "soft"):
        T, N = _sizes(rng, (4, 128), (8, 16384), 2 ** 24 // 128)
        return {"path": path, "T": 128 * T, "N": N, "beta": rng.choice([0.9, 0.95])}
    T, N = _sizes(rng, (100, 1024), (8, 64), 2 ** 16)
    return {"path": path, "T": T, "N": N, "beta": 0.95, "H": rng.choice([128, 256])}


# ----------------------------------------------------------------------------- inputs
def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    path, T, N, beta = case["path"], case["T"], case["N"], case["beta"]
    if path == "net":  # a raster of input spikes, labels, a network with weights of its own
        x = (torch.rand(T, N, 700, generator=g, device=DEVICE) < 0.015).float()
        y = torch.randint(0, 20, (N,), generator=g, device=DEVICE)
        with torch.random.fork_rng(devices=[torch.cuda.current_device()]):
            torch.manual_seed(seed)
            net = Net("auto", beta=beta, H=case["H"]).to(DEVICE)
        return {"case": case, "x": x, "y": y, "net": net, "params": list(net.parameters())}
    mean, std = CURRENTS[beta]
    I = torch.randn(T, N, generator=g, device=DEVICE).mul_(std).add_(mean)
    s = {"case": case, "I": I}
    if path == "tuned":
        s["u0"] = torch.zeros(N, device=DEVICE)
    else:
        s["u0"] = torch.rand(N, generator=g, device=DEVICE)
    if path in ("alif", "alifbox"):
        s["w0"] = torch.zeros(N, device=DEVICE)
    if path in ("layer", "tuned", "long", "fit", "alif", "affine", "soft"):
        s["gS"] = torch.randn(T, N, generator=g, device=DEVICE)
    if path in ("layer", "tuned", "fit", "alif", "affine", "soft"):
        I.requires_grad_(True)
        s["u0"].requires_grad_(True)
    names = {"fit": (beta, 1.0, U_R_FIT), "alif": (beta, RHO, Q, 1.0), "affine": (beta, GAMMA, DELTA),
             "soft": (beta,)}.get(path, ())
    s["params"] = [torch.tensor(v, device=DEVICE, requires_grad=True) for v in names]
    return s


# ----------------------------------------------------------------------------- one pass
def run(state):
    case = state["case"]
    path, beta = case["path"], case["beta"]
    if path == "net":
        logits, spikes = state["net"](state["x"])
        loss = torch.nn.functional.cross_entropy(logits, state["y"])
        return {"logits": logits.detach(), "spikes": [t.detach() for t in spikes],
                "grads": list(torch.autograd.grad(loss, state["params"]))}
    I, u0 = state["I"], state["u0"]
    if path == "infer":
        with torch.no_grad():
            return {"S": L.lif_auto(I, u0, beta)}
    if path == "long":
        U, S = L.scan_forward_v3(I, beta, 1.0, 0.0, u0, C=case["C"], K=16, repair=CONVERGE)
        dI = L.scan_backward_tiled(I, u0, U, S, state["gS"], None, beta, 1.0, 0.0, ALPHA, C=case["C"])
        return {"U": U, "S": S, "dI": dI}
    if path == "mapscan":
        U, S = L.scan_forward_v3(I, beta, 1.0, 0.0, u0, C=case["C"], K=case["K"])
        return {"U": U, "S": S}
    if path == "threelevel":
        U, S = L.scan_forward_v4(I, beta, 1.0, 0.0, u0, C=case["C"], G=case["G"])
        return {"U": U, "S": S}
    if path == "alifbox":
        C = case["C"]
        Wp = A.alif_warm_predict(I, beta, RHO, Q, 1.0, 0.0, u0, state["w0"], C)
        U, W, S = A.alif_scan_forward(I, beta, RHO, Q, 1.0, 0.0, u0, state["w0"], Wp, 0.1 * Q, C=C, K1=32,
                                      K2=32, BN=4)
        return {"U": U, "W": W, "S": S}
    ps = state["params"]
    if path == "layer":
        S = L.lif_auto(I, u0, beta)
    elif path == "tuned":
        S = L.lif_tuned(I, u0, beta, K=case["K"], repair=CONVERGE)
    elif path == "fit":
        S = F.lif_param(I, u0, *ps)
    elif path == "alif":
        S, U, W = A.alif(I, u0, state["w0"], *ps)
    elif path == "affine":
        S = AF.lif_affine(I, u0, *ps)
    else:
        S = F.lif_soft_scan(I, u0, *ps)
    grads = torch.autograd.grad(S, [I, u0] + ps, state["gS"])
    out = {"S": S.detach(), "dI": grads[0], "du0": grads[1], "dparams": list(grads[2:])}
    if path == "alif":
        out["U"], out["W"] = U, W
    return out


# ----------------------------------------------------------------------------- what a pass costs
def work(case):
    """Bytes: each call of the pass (forward, adjoint) reads its inputs and writes its outputs once.
    Operations: a step's multiply, add and compare, the surrogate and the adjoint's recurrence."""
    path, n = case["path"], case["T"] * case["N"]
    if path == "net":
        H, B, T = case["H"], case["N"], case["T"]
        rows = T * B
        fl = 2.0 * rows * H * (2 * 700 + 3 * H) + 2 * 20.0 * rows * H
        # the raster twice (forward, weight gradient); per layer currents in, spikes out, and back
        by = 4.0 * rows * (2 * 700 + H * (5 + 3 + 5 + 3))
        return {"bytes": by, "flops": fl}
    per = {"infer": (8, 3), "layer": (20, 18), "tuned": (20, 18), "long": (32, 18), "mapscan": (12, 3),
           "threelevel": (12, 3), "fit": (20, 24), "alif": (28, 36), "alifbox": (16, 6), "affine": (20, 27),
           "soft": (20, 20)}[path]
    return {"bytes": float(per[0]) * n, "flops": float(per[1]) * n}


def tolerance(case):
    """About four times what each path's outputs measured against exact(), or against the serial
    sweeps where exact() is None, over the listed cases and two dozen drawn ones."""
    path = case["path"]
    if path == "infer":
        return "exact"                      # spikes of the fp32 recurrence
    if path in ("mapscan", "threelevel", "alifbox"):
        # starts that come through maps round otherwise: states 3e-7 off (largest value 2e-6)
        return {"rel": 1.2e-6, "max": 1e-5}
    if path in ("fit", "alif", "affine", "soft"):
        # parameter gradients are sums whose terms cancel: up to 5e-6 off; dI as below
        return {"rel": 2e-5, "max": 2e-5}
    return {"rel": 1.2e-6, "max": 1e-5}     # adjoints: dI 3e-7 off (largest value 2.5e-6)


# ----------------------------------------------------------------------------- the outputs in 64 bits
def exact(case, seed):
    path, T, N = case["path"], case["T"], case["N"]
    # a spiking network's gradients in 64 bits belong to another spike train; the loops below take
    # some 25 us a step of two arrays
    if path == "net" or T > 100000:
        return None
    s = prepare(case, seed)
    f64 = torch.float64
    I, u0 = s["I"].detach(), s["u0"].detach()
    beta = float(torch.tensor(case["beta"], dtype=torch.float32))
    alif = path in ("alif", "alifbox")
    rho, q = (float(torch.tensor(v, dtype=torch.float32)) for v in (RHO, Q))
    U, V, S = torch.empty_like(I), torch.empty_like(I), torch.empty_like(I)
    W = torch.empty_like(I) if alif else None
    u, w = u0.clone(), (s["w0"].clone() if alif else None)
    ur = torch.full_like(u0, U_R_FIT if path == "fit" else 0.0)
    for t in range(T):
        v = torch.add(torch.mul(u, beta), I[t], out=V[t])
        spike = v >= (w + 1.0 if alif else 1.0)
        S[t] = spike
        if path == "affine":
            u = torch.where(spike, v * GAMMA + DELTA, v, out=U[t])
        elif path == "soft":
            u = torch.where(spike, v - 1.0, v, out=U[t])
        else:
            u = torch.where(spike, ur, v, out=U[t])
        if alif:
            w = w * rho
            w = torch.add(w, S[t] * q, out=W[t])
    if path == "infer":
        return {"S": S}
    if path in ("mapscan", "threelevel"):
        return {"U": U, "S": S}
    if path == "alifbox":
        return {"U": U, "W": W, "S": S}
    gS = s["gS"].to(f64)
    Up = torch.cat([u0[None], U[:-1]])
    Wp = torch.cat([s["w0"][None], W[:-1]]) if alif else None
    x = V.to(f64) - (1.0 + (Wp.to(f64) if alif else 0.0))
    sg = torch.sigmoid(ALPHA * x)
    sg = ALPHA * sg * (1.0 - sg)
    Sd = S.to(f64)
    lam, last = torch.empty_like(gS), torch.zeros(N, dtype=f64, device=I.device)
    if alif:
        # lw_{t-1} = (rho - q sg_t) lw_t - sg_t g_t;  lv_t = (1-s_t) beta lv_{t+1} + sg_t (g_t + q lw_t)
        lw = torch.empty_like(gS)
        a, b = rho - q * sg, sg * gS
        for t in range(T - 1, -1, -1):
            lw[t] = last
            last = a[t] * last - b[t]
        dw0, last = last, torch.zeros_like(last)
        J, b = (1.0 - Sd) * beta, sg * (gS + q * lw)
    else:
        J, b = ((1.0 - Sd) + Sd * {"affine": GAMMA, "soft": 1.0}.get(path, 0.0)) * beta, gS * sg
    for t in range(T - 1, -1, -1):
        last = torch.add(b[t], last, out=lam[t]) if t == T - 1 else torch.addcmul(b[t], J[t], last, out=lam[t])
    du0 = beta * lam[0]
    if path == "long":
        return {"U": U, "S": S, "dI": lam}
    nxt = torch.cat([lam[1:], torch.zeros_like(lam[:1])])
    dbeta = (lam * Up.to(f64)).sum()
    if path == "fit":
        dps = [dbeta, -(gS * sg).sum(), (Sd * beta * nxt).sum()]
    elif path == "alif":
        dps = [dbeta, (lw * Wp.to(f64)).sum(), (lw * Sd).sum(), -(sg * (gS + q * lw)).sum()]
    elif path == "affine":
        dps = [dbeta, (Sd * V.to(f64) * beta * nxt).sum(), (Sd * beta * nxt).sum()]
    elif path == "soft":
        dps = [dbeta]
    else:
        dps = []
    if path == "alif":
        # du0 of a detached reset: beta * lv_0
        return {"S": S, "dI": lam, "du0": du0, "dparams": dps, "U": U, "W": W}
    return {"S": S, "dI": lam, "du0": du0, "dparams": dps}
