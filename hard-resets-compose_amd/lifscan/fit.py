"""Differentiable hard-reset LIF with gradients w.r.t. the neuron parameters (beta, theta,
u_r), the interface of the reference's ``lifscan/fit.py`` (LIFParamFn, lif_param):

    dL/dbeta  = sum_t lambda_t u_{t-1}
    dL/dtheta = -sum_t gS_t sigma'(v_t - theta)           (detached reset)
    dL/du_r   = sum_t s_t beta lambda_{t+1}

with lambda_t = dL/dv_t from the adjoint.  The three sums are accumulated in fp64 inside the
adjoint kernel (lsh_lif_param_bwd), one row per block, so no [T, N] temporaries are formed.

The soft-reset layers (LIFSoftFn / lif_soft, LIFSoftScanFn / lif_soft_scan, fit.py:93-153) give
gradients for I, u0 and beta; their adjoint is lsh_soft_bwd (float64 recurrence, dbeta summed in
the kernel).  The reference's CPU prototype backend (LIFParamFnCPU) is not part of this package.
"""
import torch

from . import _native as _n
from . import hip_lif as L
from .hip_lif import _f32, _f32s, _input, _vec, _same


def _param_plan(T, N, mode):
    """lsh_lif_param_bwd's mode code and chunk for an adjoint mode name."""
    if mode == "scan":
        if N >= L.FUSED_BWD_MIN_N and T % L.FUSED_BWD_C == 0:
            return 2, L.FUSED_BWD_C
        if L.LOOKBACK_BWD and T % L.LOOKBACK_SEG == 0:
            return 3, 16
        C = L.chunked_bwd_C(T, N, min(128, L._pick_C(T, D=2)))
        return (4, 16) if L.lookback_any(N) else (1, C)
    return (4, 16) if mode == "lookback" else (0, 1)


def _param_backward(I, u0, U, S, GS, beta, theta, u_r, alpha, mode):
    """lsh_lif_param_bwd -> (Lam, sums [3] fp64)."""
    I = _input(I)
    T, N = I.shape
    u0 = _vec(u0, N, I)
    U, S, GS = (_same(a, I, nm) for a, nm in ((U, "U"), (S, "S"), (GS, "GS")))
    lib = _n.lib()
    code, C = _param_plan(T, N, mode)
    P = lib.lsh_lif_param_partials(T, N, code, C)
    if P < 0:
        raise ValueError(f"T={T} must be divisible by C={C}")
    parts = torch.zeros(max(P, 1), 3, device=I.device, dtype=torch.float64)
    Lam = torch.empty_like(I)
    ws, nbytes = None, 0
    if code == 1:
        nbytes = lib.lsh_lif_scan_bwd_workspace(T, N, C)
        ws = _n.workspace(nbytes, I.device)
    elif code >= 3:
        nbytes = lib.lsh_lif_scan_lookback_any_bwd_workspace(T, N)
        ws = _n.workspace(nbytes, I.device)
    with _n.on_device(I):
        _n.check(lib.lsh_lif_param_bwd(
            _n.ptr(I), _n.ptr(u0), _n.ptr(U), _n.ptr(S), _n.ptr(GS), _n.ptr(Lam), _n.ptr(parts), T, N,
            _f32(beta), _f32(theta), _f32(u_r), _f32(alpha), code, C, _n.ptr(ws), nbytes,
            _n.stream_of(I)), "lsh_lif_param_bwd")
    if code >= 3:
        L._note_lookback(ws)
    return Lam, parts.sum(0)


class LIFParamFn(torch.autograd.Function):
    """S = LIF(I; u0, beta, theta, u_r) with gradients for I, u0 and the three parameters
    (fit.py:15-48).  fwd_mode / bwd_mode: "serial" or "scan", or lif_param's own choices (choose: True,
    or the three parameters' values already read)."""

    @staticmethod
    def forward(ctx, I, u0, beta, theta, u_r, alpha, fwd_mode, bwd_mode, K, choose=False):
        b, th, ur = choose if isinstance(choose, tuple) else _f32s(beta, theta, u_r)
        I = I.contiguous()
        T, N = I.shape
        route = L._auto_route(T, N, b) if choose and L._layer_ok(N) and T > 0 else None
        ctx.cfg = (b, th, ur, float(alpha), "lookback" if route else bwd_mode)
        # lif_param's own choice: the exact forward's bits are the serial one's, so the states before
        # every 32 rows are kept instead of U
        if route == (0, 0):
            S, ST = L._layer_forward(I, b, th, ur, u0)
            ctx.save_for_backward(I, u0, ST)
            ctx.recompute = True
            return S
        if choose:
            U, S = L._auto_forward(I, b, th, ur, u0, K, 0, route, fwd_mode)
        elif fwd_mode == "scan":
            U, S = L.scan_forward_auto(I, b, th, ur, u0, K=K)
        else:
            U, S = L.serial_forward_auto(I, b, th, ur, u0)
        ctx.save_for_backward(I, u0, U, S)
        ctx.recompute = False
        return S

    @staticmethod
    def backward(ctx, gS):
        b, th, ur, alpha, bwd_mode = ctx.cfg
        if ctx.recompute:
            I, u0, ST = ctx.saved_tensors
            lam, sums = L._layer_backward(I, ST, gS.contiguous(), b, th, ur, alpha, True)
        else:
            I, u0, U, S = ctx.saved_tensors
            lam, sums = _param_backward(I, u0, U, S, gS.contiguous(), b, th, ur, alpha, bwd_mode)
        sums = sums.float()
        need = ctx.needs_input_grad  # a gradient only for the parameters given as tensors
        du0 = b * lam[0] if ctx.needs_input_grad[1] else None
        return (lam, du0, sums[0] if need[2] else None, -sums[1] if need[3] else None,
                b * sums[2] if need[4] else None, None, None, None, None, None)


def lif_param(I, u0, beta, theta, u_r, alpha=4.0, mode="auto", K=16):
    """fit.py:51-57: mode "auto" picks serial / scan per pass from (N, T).  Parameters may be
    0-d tensors or floats; floats go to the kernels as they are (the reference wraps them in
    device tensors and reads them back: the same fp32 values, one synchronizing copy more)."""
    T, N = I.shape
    choose = mode == "auto"
    if choose:
        L._check_auto_args(T, N, K, 0)
        fwd, bwd = L.auto_modes(N, T)
        fwd, bwd = L._auto_fwd(fwd, N, T), L._auto_bwd(bwd, N, T)
        u0v = L._cpp_u0(I, u0, alpha) if L._layer_ok(N) else None
        if u0v is not None:  # the same kernels as LIFParamFn's, from C++
            b, th, ur = choose = _f32s(beta, theta, u_r)
            route = L._auto_route(T, N, b, L._wants_grad(I, u0v, beta, theta, u_r))
            if route is not None:
                return _n.ops().lif_layer(I, u0v, *map(L._grad_param, (beta, theta, u_r)), b, th, ur,
                                          float(alpha), L._wait_header(I.device), *route)
    else:
        fwd = bwd = mode
    return LIFParamFn.apply(I, u0, beta, theta, u_r, alpha, fwd, bwd, K, choose)


class LIFSoftFn(torch.autograd.Function):
    """Soft (subtractive) reset LIF, serial forward; gradients for I, u0, beta (fit.py:93-114)."""

    @staticmethod
    def forward(ctx, I, u0, beta, theta, alpha):
        from . import hip_soft as TS
        b, th = _f32s(beta, theta)
        I = I.contiguous()
        U, S = TS.soft_serial_forward(I, b, th, u0)
        ctx.save_for_backward(I, u0, U)
        ctx.cfg = (b, th, float(alpha))
        return S

    @staticmethod
    def backward(ctx, gS):
        from . import hip_soft as TS
        I, u0, U = ctx.saved_tensors
        b, th, alpha = ctx.cfg
        need_b = ctx.needs_input_grad[2]
        lam, db = TS._soft_backward(I, u0, U, gS.contiguous(), b, th, alpha, need_b)
        du0 = b * lam[0] if ctx.needs_input_grad[1] else None
        return lam, du0, (db.float().reshape(()) if need_b else None), None, None


def lif_soft(I, u0, beta, theta=1.0, alpha=4.0):
    """fit.py:117-118."""
    return LIFSoftFn.apply(I, u0, beta, theta, alpha)


class LIFSoftScanFn(torch.autograd.Function):
    """Soft-reset LIF with the exact soft scan forward (mode "scan", the reference's default
    repair = 0) or the serial forward; the adjoint is the float64 recurrence in both modes (the
    reference: FFT convolution for "scan", the fp32 serial sweep otherwise); gradients for I,
    u0, beta (fit.py:121-149)."""

    @staticmethod
    def forward(ctx, I, u0, beta, theta, alpha, mode, C, K):
        from . import hip_soft as TS
        b, th = _f32s(beta, theta)
        I = I.contiguous()
        if mode == "scan":
            U, S = TS.soft_scan_forward(I, b, th, u0, C=C, K=K)
        else:
            U, S = TS.soft_serial_forward(I, b, th, u0)
        ctx.save_for_backward(I, u0, U)
        ctx.cfg = (b, th, float(alpha))
        return S

    @staticmethod
    def backward(ctx, gS):
        from . import hip_soft as TS
        I, u0, U = ctx.saved_tensors
        b, th, alpha = ctx.cfg
        need_b = ctx.needs_input_grad[2]
        lam, db = TS._soft_backward(I, u0, U, gS.contiguous(), b, th, alpha, need_b)
        du0 = b * lam[0] if ctx.needs_input_grad[1] else None
        return (lam, du0, (db.float().reshape(()) if need_b else None), None, None, None, None,
                None)


def lif_soft_scan(I, u0, beta, theta=1.0, alpha=4.0, mode="scan", C=128, K=32):
    """fit.py:152-153."""
    from . import hip_affine as AF
    from . import hip_soft as TS
    u0v = AF._cpp_layer_u0(I, u0, mode, C, K, theta, alpha)
    if u0v is not None:  # the same kernels as LIFSoftScanFn's, from C++
        b, th = _f32s(beta, theta)
        return AF._cpp_layer(I, u0v, (beta, None, None), (b, th, 1.0, -th, float(alpha)), True, mode, C,
                             K, 0, TS._soft_C(*I.shape))
    return LIFSoftScanFn.apply(I, u0, beta, theta, alpha, mode, C, K)
