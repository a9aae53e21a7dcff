"""Point-source lensing on the GPU (reference: src/caustics/point_source.py).

``mag_point_source(w, nlenses=2, roots_itmax=2500, roots_compensated=False, **params)``
(:1762-1830) runs in one fused HIP kernel per evaluation: parameter map and x_cm
shift, FP64 coefficients, all-roots solve, lens-equation filter (1e-6), sum of
1/|det J|.  Where a gradient is needed (torch.autograd) the same kernel pushes
implicit-derivative tangents of w and of every lens parameter through det J and keeps
that Jacobian; the backward pass scales it and sums it over broadcast parameters.

``lens_eq`` and ``lens_eq_det_jac`` (:1536-1580) take lens-frame parameters
(a, e1[, e2, r3]) exactly as in the reference and are elementwise tensor expressions.

``images_point_source`` and ``images_point_source_sequential`` (:1652-1759, the
reference's private ``_images_point_source`` and ``_images_point_source_sequential``)
return the images and the real-image mask for lens-frame source positions and
lens-frame parameters; the sequential form warm-starts each position from the previous
one's roots, so that row j follows one image along the sequence.  They return no
gradients (``mag_point_source`` and ``ehrlich_aberth`` do).
"""
import ctypes

import numpy as np
import torch

from . import _lib

__all__ = [
    "mag_point_source",
    "images_point_source",
    "images_point_source_sequential",
    "lens_eq",
    "lens_eq_det_jac",
    "critical_and_caustic_curves",
    "PARAM_NAMES",
]

PARAM_NAMES = {1: (), 2: ("s", "q"), 3: ("s", "q", "q3", "r3", "psi")}


def _mode_id(roots_compensated, mode):
    if mode is None:
        mode = "fp64_comp" if roots_compensated else "fp64"
    return _lib.MODES[mode]


def _tensor(x, like=None):
    if isinstance(x, torch.Tensor):
        return x
    return torch.as_tensor(np.asarray(x), device="cuda")


def _prepare(w, nlenses, params):
    w = _tensor(w)
    if not w.is_complex():
        w = w.to(torch.float64)
    w = _lib.on_device(w, torch.complex128)
    names = PARAM_NAMES[nlenses]
    missing = [n for n in names if n not in params]
    if missing:
        raise ValueError(f"nlenses={nlenses} needs parameters {names}; missing {missing}")
    ps = [_lib.on_device(_tensor(params[n]), torch.float64) for n in names]
    return w, ps


# A backward pass scales and reduces the Jacobian that the forward pass kept, 8 bytes a position
# for each parameter that requires a gradient (16 for the position itself).  Solving the roots
# again instead costs 8 times as much (512,000 binary epochs: 93 against 11 us on one MI355X)
# and no memory, so that is what a call does whose Jacobian would exceed this many bytes, or
# would leave less than half of the card free (the Jacobians of one graph add up), or cannot be
# allocated.
JACOBIAN_MAX_BYTES = 4 << 30
# Asking for the free memory takes 5 us, and up to 20 where the autograd engine's thread is slow
# to wake, so it is asked once for this many bytes of Jacobians handed out.
JACOBIAN_ASK_BYTES = 1 << 30
# device index -> bytes that may be handed out before the next question (threads that race for it
# hand out at most that much each)
_jacobian_credit = {}
_saved_tensor_hooks = torch._C._autograd._top_saved_tensors_default_hooks


def _half_free(need, device):
    """need bytes out of the half of the card that Jacobians may take: what the driver has free,
    and what torch's allocator holds unused."""
    free, total = torch.cuda.mem_get_info(device)
    if free - need >= total // 2:
        return True
    st = torch.cuda.memory_stats_as_nested_dict(device)
    held = st["reserved_bytes"]["all"]["current"] - st["allocated_bytes"]["all"]["current"]
    return free + held - need >= total // 2


def kept_jacobian(planes, N, device, limit):
    """Memory for the (planes, N) Jacobian of a forward pass, or None where the backward pass is
    to solve again."""
    need = 8 * planes * N
    if need > limit:
        return None
    dev = device.index
    credit = _jacobian_credit.get(dev, 0)
    # Where hooks take what is saved, the sizes decide alone: activation checkpointing runs the
    # forward pass again, when other memory is free, and requires that the same is saved (and
    # holds one segment's Jacobians at a time); save_on_cpu takes them off the card.
    if need > credit and _saved_tensor_hooks(True) is None:
        credit = need + JACOBIAN_ASK_BYTES
        if not _half_free(credit, device):
            return None
    _jacobian_credit[dev] = max(credit - need, 0)
    try:
        return torch.empty((planes, N), dtype=torch.float64, device=device)
    except torch.OutOfMemoryError:
        return None


def jacobian_vjp(jac, nw, rows, g, want_w, want_p):
    """Backward pass of the kept Jacobian jac (nw + np, N) for cotangents g (N,): (g_w (N,)
    complex or None, g_p (np, N / rows) sums over rows of consecutive items or None).  The np
    planes are those of the parameters that require a gradient, in their order."""
    npl, N = jac.shape
    n_p = npl - nw
    g_w = torch.empty(N, dtype=torch.complex128, device=jac.device) if want_w else None
    g_p = None
    if want_p and n_p:
        shape = (n_p, N // rows)
        g_p = (torch.empty if N else torch.zeros)(shape, dtype=torch.float64, device=jac.device)
    L = _lib.lib()
    wsb = L.caus_jacobian_workspace_bytes(n_p, N, rows)
    ws = torch.empty(wsb // 8, dtype=torch.float64, device=jac.device) if wsb > 0 else None
    rc = L.caus_jacobian_vjp(_lib.stream_ptr(), _lib.ptr(jac), N, nw, n_p, rows, _lib.ptr(g),
                             _lib.ptr(g_w), _lib.ptr(g_p), _lib.ptr(ws), wsb)
    _lib.check(rc, "caus_jacobian_vjp")
    return g_w, g_p


def _param_rows(shape, ps):
    """Items per parameter row when every parameter is broadcast over the same trailing
    dimensions of shape (the shape of the items), else 1 (a row for each item)."""
    N = 1
    for n in shape:
        N *= n
    if all(p.numel() == 1 for p in ps):
        return max(N, 1)
    first = (1,) * (len(shape) - ps[0].dim()) + tuple(ps[0].shape)
    if any((1,) * (len(shape) - p.dim()) + tuple(p.shape) != first for p in ps[1:]):
        return 1
    per, d = 1, len(shape)
    while d > 0 and first[d - 1] == 1:
        d -= 1
        per *= shape[d]
    return per if first[:d] == tuple(shape[:d]) and N else 1


class _MagPointSource(torch.autograd.Function):
    @staticmethod
    def forward(ctx, nlenses, itmax, mode, need, w, *ps):
        shape = torch.broadcast_tensors(w, *ps)[0].shape
        wf = w.expand(shape).contiguous().reshape(-1)
        N = wf.numel()
        P = len(ps)
        per = _param_rows(shape, ps) if P else 1
        if per > 1 or N == 1:
            cols = [p.reshape(-1) for p in ps]
        else:
            cols = [p.expand(shape).reshape(-1) for p in ps]
        mag = torch.empty(N, dtype=torch.float64, device=w.device)
        jac, nw, planes, wrt = None, 0, 0, []
        if need:
            nw = 2 if ctx.needs_input_grad[4] else 0
            wrt = [k for k, g in enumerate(ctx.needs_input_grad[5:]) if g]
            planes = (3 if nw else 0) + sum([4 << k for k in wrt])
            jac = kept_jacobian(nw + len(wrt), N, w.device, JACOBIAN_MAX_BYTES)
        rc = _lib.lib().caus_mag_point_source_jac_planes(
            _lib.stream_ptr(), nlenses, _lib.ptr(wf), N, *_lib.columns(cols), per,
            _lib.ptr(mag), _lib.ptr(jac), planes, itmax, mode)
        _lib.check(rc, "caus_mag_point_source_jac_planes")
        if jac is not None:
            ctx.save_for_backward(jac)
        elif need:
            prm = torch.stack([c.expand(N // per) for c in cols], -1).contiguous() if P else None
            ctx.save_for_backward(None, wf, prm)
        ctx.meta = (nlenses, itmax, mode, shape, per, w.shape, [p.shape for p in ps], nw, wrt)
        return mag.reshape(shape)

    @staticmethod
    def backward(ctx, g):
        nlenses, itmax, mode, shape, per, wshape, pshapes, nw, wrt = ctx.meta
        jac, *again = ctx.saved_tensors
        P = len(pshapes)
        want_w, want_p = ctx.needs_input_grad[4], any(ctx.needs_input_grad[5:])
        gf = _lib.resolved(g.expand(shape).contiguous().reshape(-1).to(torch.float64))
        if jac is not None:
            g_w, g_p = jacobian_vjp(jac, nw, per, gf, want_w, want_p)
            pshape = shape if per == 1 else None   # summed over the rows already
        else:
            wf, prm = again
            N = wf.numel()
            wrt = range(P)
            pstride = P if P and prm.shape[0] > 1 else 0
            if pstride and per > 1:
                prm = prm.repeat_interleave(per, 0)
            mag = torch.empty(N, dtype=torch.float64, device=wf.device)
            g_w = torch.empty(N, dtype=torch.complex128, device=wf.device)
            g_p = torch.empty((N, max(P, 1)), dtype=torch.float64, device=wf.device)
            rc = _lib.lib().caus_mag_point_source_vjp(
                _lib.stream_ptr(), nlenses, _lib.ptr(wf), N, _lib.ptr(prm), pstride, _lib.ptr(gf),
                _lib.ptr(mag), _lib.ptr(g_w), _lib.ptr(g_p), None, itmax, mode)
            _lib.check(rc, "caus_mag_point_source_vjp")
            g_p = g_p.t()
            pshape = shape
        gw = g_w.reshape(shape).sum_to_size(wshape) if want_w else None
        gps = [None] * P
        for k, row in zip(wrt, g_p.unbind(0) if g_p is not None else ()):
            if ctx.needs_input_grad[5 + k]:
                gps[k] = (row.reshape(pshapes[k]) if pshape is None else
                          row.reshape(shape).sum_to_size(pshapes[k]))
        return (None, None, None, None, gw, *gps)


def mag_point_source(w, nlenses=2, roots_itmax=2500, roots_compensated=False, mode=None,
                     **params):
    """Point-source magnification at source positions ``w`` (complex), in the frame of
    the reference: origin at the centre of mass of lenses 1-2, which lie on the real
    axis.  Parameters: ``s, q`` (nlenses=2) or ``s, q, q3, r3, psi`` (nlenses=3); each
    may be a float or a tensor broadcastable against ``w``.  Differentiable in ``w``
    and every parameter.  ``mode``: "fp64" (default), "fp64_comp" (= roots_compensated)
    or "cf32"."""
    if nlenses not in (1, 2, 3):
        raise ValueError("`nlenses` has to be set to be <= 3.")
    w, ps = _prepare(w, nlenses, params)
    need = torch.is_grad_enabled() and (w.requires_grad or any(p.requires_grad for p in ps))
    return _MagPointSource.apply(nlenses, int(roots_itmax), _mode_id(roots_compensated, mode),
                                 need, w, *ps)


_DEGREE = {1: 2, 2: 5, 3: 10}


def _as64(v):
    """v on the device in 64-bit precision (float64, or complex128 when complex);
    torch.as_tensor alone makes python floats and lists float32."""
    if torch.is_tensor(v):
        return v.to(device="cuda", dtype=torch.complex128 if v.is_complex() else torch.float64)
    a = np.asarray(v)
    return torch.as_tensor(a.astype(np.complex128 if np.iscomplexobj(a) else np.float64),
                           device="cuda")


def _lens_rows(nlenses, shape, params):
    """Lens-frame parameter rows (a, e1) or (a, e1, e2, Re r3, Im r3) broadcast to
    `shape` (the source positions' batch shape, sequences flattened)."""
    if nlenses == 1:
        return None
    names = ("a", "e1") if nlenses == 2 else ("a", "e1", "e2", "r3")
    cols = []
    for n in names:
        v = params[n]
        if n == "r3":
            # python floats and complexes straight to 64-bit (as_tensor would make float32)
            v = torch.as_tensor(v, dtype=torch.complex128, device="cuda")
            cols += [v.real, v.imag]
        else:
            v = (v.to(device="cuda", dtype=torch.float64) if torch.is_tensor(v)
                 else torch.as_tensor(v, dtype=torch.float64, device="cuda"))
            cols.append(v)
    cols = [c.expand(shape).reshape(-1) for c in cols]
    return torch.stack(cols, -1).contiguous()


def _images(w, nlenses, itmax, mode, z_init, sequential, params):
    L = _lib.lib()
    n = _DEGREE[nlenses]
    B, N = w.shape
    lens = _lens_rows(nlenses, (B,) if sequential else (B, N), params)
    if lens is not None and not sequential:
        lens = lens.reshape(B * N, -1)
    z = torch.empty((B, N, n), dtype=torch.complex128, device="cuda")
    mask = torch.empty((B, N, n), dtype=torch.uint8, device="cuda")
    status = torch.empty((B, N), dtype=torch.uint8, device="cuda")
    zi = None
    if z_init is not None:
        zi = (_lib.on_device(z_init, torch.complex128) if torch.is_tensor(z_init)
              else torch.as_tensor(np.asarray(z_init, np.complex128), device="cuda"))
        zi = zi.reshape(n, B, N).permute(1, 2, 0).contiguous()
    # independent positions: one lens row per position, addressed as B*N sequences of 1
    Bc, Nc = (B, N) if sequential else (B * N, 1)
    rc = L.caus_images_point_source(_lib.stream_ptr(), nlenses, _lib.ptr(w), Bc, Nc,
                                    _lib.ptr(lens), 0 if lens is None else lens.shape[1],
                                    _lib.ptr(zi), _lib.ptr(z), _lib.ptr(mask), _lib.ptr(status),
                                    int(itmax), mode, 1 if sequential else 0)
    _lib.check(rc, "caus_images_point_source")
    return z, mask.bool(), status


def images_point_source(w, nlenses=2, roots_itmax=2500, roots_compensated=False,
                        custom_init=False, z_init=None, mode=None, **params):
    """Images (n, *w.shape) complex and the real-image mask (|lens_eq(z) - w| < 1e-6) of
    lens-frame source positions w; parameters a, e1 (nlenses=2) or a, e1, e2, r3
    (nlenses=3), floats or tensors broadcastable against w.  custom_init with z_init
    (n, *w.shape) starts the solver from those roots (point_source.py:1652-1709)."""
    if nlenses not in (1, 2, 3):
        raise ValueError("`nlenses` has to be set to be <= 3.")
    w = (_lib.on_device(w, torch.complex128) if torch.is_tensor(w)
         else torch.as_tensor(np.asarray(w, np.complex128), device="cuda"))
    shape = w.shape
    wf = w.reshape(1, -1).contiguous()
    prm = {k: (_as64(v).expand(shape).reshape(1, -1) if torch.is_tensor(v) or np.ndim(v) else v)
           for k, v in params.items()}
    z, mask, _ = _images(wf, nlenses, roots_itmax, _mode_id(roots_compensated, mode),
                         z_init if custom_init else None, False, prm)
    n = _DEGREE[nlenses]
    return (z.reshape(*shape, n).movedim(-1, 0), mask.reshape(*shape, n).movedim(-1, 0))


def images_point_source_sequential(w, nlenses=2, roots_itmax=2500, roots_compensated=False,
                                   mode=None, **params):
    """Images along a sequence of lens-frame source positions w (N,) solved in order, each
    position started from the previous one's roots (point_source.py:1711-1759): returns
    z (n, N) and the mask (n, N).  A 2-D w (B, N) runs B sequences at once, with
    parameters of shape (B,) or scalars, and returns (B, n, N)."""
    if nlenses not in (1, 2, 3):
        raise ValueError("`nlenses` has to be set to be <= 3.")
    w = (_lib.on_device(w, torch.complex128) if torch.is_tensor(w)
         else torch.as_tensor(np.asarray(w, np.complex128), device="cuda"))
    one = w.dim() == 1
    w2 = (w.reshape(1, -1) if one else w).contiguous()
    B = w2.shape[0]
    prm = {k: (_as64(v).reshape(-1) if torch.is_tensor(v) or np.ndim(v) else v)
           for k, v in params.items()}
    z, mask, _ = _images(w2, nlenses, roots_itmax, _mode_id(roots_compensated, mode), None,
                         True, {k: (v if not torch.is_tensor(v) else v.expand(B)) for k, v in
                                prm.items()})
    z, mask = z.permute(0, 2, 1), mask.permute(0, 2, 1)   # (B, n, N)
    return (z[0], mask[0]) if one else (z, mask)


def _lens_terms(z, nlenses, params):
    zb = torch.conj(z)
    if nlenses == 1:
        return [(1.0, 0.0)], zb
    a, e1 = params["a"], params["e1"]
    if nlenses == 2:
        return [(e1, a), (1.0 - e1, -a)], zb
    e2, r3 = params["e2"], params["r3"]
    r3 = r3 if isinstance(r3, torch.Tensor) else torch.as_tensor(complex(r3), device=z.device,
                                                                 dtype=torch.complex128)
    return [(e1, a), (e2, -a), (1.0 - e1 - e2, r3)], zb


def lens_eq(z, nlenses=2, **params):
    """w = z - sum_j e_j / (conj z - conj r_j) with lens-frame parameters
    (point_source.py:1536-1556)."""
    z = _tensor(z).to(torch.complex128)
    terms, zb = _lens_terms(z, nlenses, params)
    out = z
    for e, r in terms:
        r_c = torch.conj(r) if isinstance(r, torch.Tensor) else r
        out = out - e / (zb - r_c)
    return out


def lens_eq_det_jac(z, nlenses=2, **params):
    """det J = 1 - |sum_j e_j / (conj z - conj r_j)^2|^2 (point_source.py:1558-1580)."""
    z = _tensor(z).to(torch.complex128)
    terms, zb = _lens_terms(z, nlenses, params)
    K = 0
    for e, r in terms:
        r_c = torch.conj(r) if isinstance(r, torch.Tensor) else r
        K = K + e / (zb - r_c) ** 2
    return 1.0 - torch.abs(K) ** 2


def _critical_coeffs(phi, nlenses, a, e1, e2=None, r3=None):
    """Highest-first coefficients of prod_j (z - r_j)^2 exp(-i phi) - sum_j e_j
    prod_{k!=j} (z - r_k)^2, the critical-curve polynomial (point_source.py:1482-1534)."""
    x = torch.exp(-1j * phi) * torch.ones_like(a)   # (B, npts)
    one = torch.ones_like(x)
    if nlenses == 2:
        return torch.stack([x, 0 * x, -2 * a**2 * x - 1.0, (-4 * a * e1 + 2 * a) * one,
                            a**4 * x - a**2], -1)
    p = [x, -2 * x * r3, -2 * a**2 * x - 1 + x * r3**2,
         4 * a**2 * x * r3 - 2 * a * e1 + 2 * a * e2 + 2 * e1 * r3 + 2 * e2 * r3,
         (a**4 * x - 3 * a**2 * e1 - 3 * a**2 * e2 + 2 * a**2 - 2 * a**2 * x * r3**2
          + 4 * a * e1 * r3 - 4 * a * e2 * r3 - e1 * r3**2 - e2 * r3**2),
         (-2 * a**4 * x * r3 + 2 * a**2 * e1 * r3 + 2 * a**2 * e2 * r3 - 2 * a * e1 * r3**2
          + 2 * a * e2 * r3**2),
         (a**4 * e1 + a**4 * e2 - a**4 + a**4 * x * r3**2 - a**2 * e1 * r3**2
          - a**2 * e2 * r3**2) * one]
    return torch.stack(p, -1)


def critical_and_caustic_curves(npts=200, nlenses=2, **params):
    """Critical curves and caustics, each (n_curves, npts) complex, in the frame of the
    reference API (point_source.py:1582-1649): roots of the critical-curve polynomial
    on a grid of phi (GPU solver), continued along phi with match_points, mapped through
    the lens equation and shifted by x_cm (HIP kernels).  Parameters may also be
    arrays of length B (s, and any of the others), giving (B, n_curves, npts)."""
    phi = torch.linspace(-np.pi, np.pi, npts, dtype=torch.float64, device="cuda")
    if nlenses == 1:
        return torch.exp(-1j * phi), torch.zeros(npts, dtype=torch.complex128, device="cuda")
    names = PARAM_NAMES[nlenses]
    if any(isinstance(params[k], torch.Tensor) and _differentiated(params[k]) for k in names):
        return _curves_tensor(phi, nlenses, [params[k] for k in names])
    # numbers go to the kernels by value
    vals = [v if isinstance(v, torch.Tensor) else np.asarray(v) for v in
            (params[k] for k in names)]
    batch = vals[0].ndim > 0
    cols = [None if isinstance(v, np.ndarray) and v.ndim == 0 else
            _lib.resolved(torch.as_tensor(v, device="cuda").to(torch.float64)).reshape(-1)
            for v in vals]
    B = torch.broadcast_shapes(*[(1,) if c is None else c.shape for c in cols])[0]
    if B != (1 if cols[0] is None else cols[0].numel()):
        raise RuntimeError(f"{names[0]} has to have the length of the batch, {B}")
    P = len(cols)
    n = _DEGREE_CRITICAL[nlenses]
    crit = torch.empty((B, n, npts), dtype=torch.complex128, device="cuda")
    caus = torch.empty_like(crit)
    L = _lib.lib()
    wsb = L.caus_critical_curves_workspace_bytes(nlenses, B, npts)
    ws = torch.empty((wsb + 7) // 8, dtype=torch.float64, device="cuda")
    rc = L.caus_critical_curves(
        _lib.stream_ptr(), nlenses,
        (ctypes.c_void_p * P)(*[None if c is None else c.data_ptr() for c in cols]),
        (ctypes.c_int64 * P)(*[0 if c is None or c.numel() == 1 else c.stride(0) for c in cols]),
        (ctypes.c_double * P)(*[float(v) if c is None else 0.0 for v, c in zip(vals, cols)]),
        B, _lib.ptr(phi), npts, _lib.ptr(crit), _lib.ptr(caus), _lib.ptr(ws), wsb, 2000)
    _lib.check(rc, "caus_critical_curves")
    return (crit, caus) if batch else (crit[0], caus[0])


_DEGREE_CRITICAL = {2: 4, 3: 6}


def _differentiated(x):
    """Whether a derivative with respect to x is recorded, or x carries a forward-mode tangent
    (which the root solver refuses; a kernel would drop it)."""
    return ((torch.is_grad_enabled() and x.requires_grad)
            or torch.autograd.forward_ad.unpack_dual(x).tangent is not None)


def _curves_tensor(phi, nlenses, params):
    """critical_and_caustic_curves as tensor expressions around the root solver and the
    continuation, for differentiated parameters (a gradient flows through the explicit
    dependence of the map and the shift on them)."""
    from .ehrlich_aberth_primitive import poly_roots

    npts = phi.numel()
    vals = [torch.as_tensor(np.asarray(v) if not isinstance(v, torch.Tensor) else v,
                            device="cuda").to(torch.float64) for v in params]
    batch = vals[0].dim() > 0
    vals = [v.reshape(-1, 1) for v in vals]
    s, q = vals[0], vals[1]
    a = 0.5 * s
    x_cm = a * (1 - q) / (1 + q)
    if nlenses == 2:
        e1 = 1 / (1 + q)
        coeffs = _critical_coeffs(phi[None, :], 2, a, e1)
        lf = dict(a=a, e1=e1)
    else:
        q3, r3m, psi = vals[2], vals[3], vals[4]
        e1 = q / (1 + q + q3)
        e2 = q * e1
        r3 = r3m * torch.exp(1j * psi)
        coeffs = _critical_coeffs(phi[None, :], 3, a, e1, e2, r3)
        lf = dict(a=a, e1=e1, e2=e2, r3=r3)
    z = poly_roots(coeffs).contiguous()            # (B, npts, n)
    B, _, n = z.shape
    zc = torch.empty_like(z)
    rc = _lib.lib().caus_match_chain(_lib.stream_ptr(), _lib.ptr(z), _lib.ptr(zc), npts, n, B)
    _lib.check(rc, "caus_match_chain")
    zc = zc.transpose(1, 2)                        # (B, n, npts)
    lfb = {k: (v[:, :, None] if isinstance(v, torch.Tensor) else v) for k, v in lf.items()}
    za = lens_eq(zc, nlenses=nlenses, **lfb)
    zc = zc - x_cm[:, :, None]
    za = za - x_cm[:, :, None]
    if not batch:
        return zc[0], za[0]
    return zc, za
