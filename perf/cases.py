"""Timed cases: what a program built on caustics_amd calls, at the sizes it calls it with.

``listed()`` names the cases, ``draw(rng)`` gives further ones of the same ranges,
``prepare(case, seed)`` makes what the program holds before the call, ``run(state)`` is one
pass through the public entry points and returns whole outputs (values and gradients),
``work(case)`` counts what a pass cannot do without, and ``exact(case, seed)`` gives the
same outputs in plain 64-bit numpy / torch where that is possible in seconds.

Inputs follow the distributions of caustics_amd.workloads (lens separations, mass ratios,
trajectories and source radii log-uniform over the ranges of microlensing events).
"""
import math

import numpy as np
import torch

import caustics_amd as ca

DEV = "cuda"
LENS_NAMES = {2: ("s", "q"), 3: ("s", "q", "q3", "r3", "psi")}
DEGREE = {2: 5, 3: 10}


def listed():
    return [
        # one lens plotted or inspected: its critical curve and caustic, the default 200
        # points (a call whose cost is latency)
        dict(name="caustic_curves", kind="curves", nl=2, npts=200),
        # a map of point-source magnifications of one binary lens
        dict(name="point_source_binary", kind="ps", nl=2, n=10000, grad=False),
        # point-source magnifications of a triple lens with gradients, an odd count
        dict(name="point_source_triple_grad", kind="ps", nl=3, n=50001, grad=True),
        # one binary light curve with its gradient: the step of a single chain or optimiser
        dict(name="lightcurve_one_grad", kind="lc", nl=2, l=1, t=1500),
        # a batch of binary light curves with gradients: many chains, or a grid search
        dict(name="lightcurve_batch_grad", kind="lc", nl=2, l=256, t=2000),
        # the root operator as the reference binds it (default initial estimates, so its
        # root order), with the gradient to the coefficients
        dict(name="roots_deg5_grad", kind="roots", nl=2, n=262144, init="reference", grad=True),
        # a large batch of triple-lens polynomials from complex initial estimates
        dict(name="roots_deg10", kind="roots", nl=3, n=262144, init="complex", grad=False),
        # one extended source, the call the reference's function makes (its default limb
        # resolution, uniform disk)
        dict(name="extended_one", kind="ext", nl=2, sets=1, epochs=1, npts=150, ld=False,
             grad=False),
        # a limb-darkened light curve over an event: mag() decides per epoch between the
        # hexadecapole value and the contour, default resolution
        dict(name="mag_event", kind="mag", n=500, npts_max=200, ragged=False, grad=False),
        # an inference batch of limb-darkened binary sources, half of them near a caustic,
        # uneven limb resolutions, with gradients
        dict(name="mag_batch_grad", kind="mag", n=4096, npts_max=4096, ragged=True, grad=True),
        # triple-lens limb-darkened light curves through a caustic, uneven limb
        # resolutions, with gradients
        dict(name="extended_triple_grad", kind="ext", nl=3, sets=16, epochs=1500, npts=4096,
             ld=True, grad=True),
        # a whole inference step: parallax trajectory, magnification, flux-marginalised
        # likelihood of two observatories, gradients to every parameter
        dict(name="inference_step", kind="infer", l=64, t=1500),
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["curves", "ps", "ps", "lc", "lc", "roots", "roots", "ext", "ext", "mag",
                       "mag", "infer"])
    nl = rng.choice([2, 3])
    grad = rng.choice([False, True])
    if kind == "curves":
        return dict(kind=kind, nl=nl, npts=_size(rng, 50, 400))
    if kind == "ps":
        return dict(kind=kind, nl=nl, n=_size(rng, 1000, 60000), grad=grad)
    if kind == "lc":
        l = _size(rng, 1, 256)
        return dict(kind=kind, nl=2, l=l, t=_size(rng, 200, 2000))
    if kind == "roots":
        return dict(kind=kind, nl=nl, n=_size(rng, 1000, 262144),
                    init=rng.choice(["reference", "complex"]), grad=grad)
    if kind == "ext":
        big = rng.random() < 0.5
        return dict(kind=kind, nl=nl, sets=_size(rng, 1, 12) if big else 1,
                    epochs=_size(rng, 200, 1400) if big else _size(rng, 1, 60),
                    npts=rng.choice([1024, 4096]) if big else rng.choice([150, 200, 333, 512]),
                    ld=True if big else rng.choice([False, True]), grad=grad)
    if kind == "mag":
        ragged = rng.random() < 0.5
        return dict(kind=kind, n=_size(rng, 50, 4000), ragged=ragged,
                    npts_max=rng.choice([1024, 4096]) if ragged else rng.choice([200, 256, 501]),
                    grad=grad)
    return dict(kind="infer", l=_size(rng, 1, 128), t=_size(rng, 300, 1500))


# ---- inputs -------------------------------------------------------------------------
def _loguniform(g, lo, hi, n):
    return 10.0 ** g.uniform(np.log10(lo), np.log10(hi), n)


def _lenses(g, n, nl):
    p = {"s": _loguniform(g, 0.3, 3.0, n), "q": _loguniform(g, 1e-4, 1.0, n)}
    if nl == 3:
        p["r3"] = g.uniform(0.3, 2.0, n)
        p["psi"] = g.uniform(0.0, 2 * np.pi, n)
        p["q3"] = _loguniform(g, 1e-4, 1e-1, n)
    return p


def _frame(p, nl, np_=np):
    """Masses, positions and the shift of the lens frame, broadcast over the items."""
    s, q = p["s"], p["q"]
    a = 0.5 * s
    x_cm = a * (1 - q) / (1 + q)
    if nl == 2:
        e1 = 1 / (1 + q)
        return [e1, 1 - e1], [a + 0j, -a + 0j], x_cm
    e1 = q / (1 + q + p["q3"])
    e2 = q * e1
    r3 = p["r3"] * np_.exp(1j * p["psi"])
    return [e1, e2, 1 - e1 - e2], [a + 0j, -a + 0j, r3], x_cm


def _disk(g, n, radius=2.0):
    return radius * np.sqrt(g.uniform(0, 1, n)) * np.exp(2j * np.pi * g.uniform(0, 1, n))


def _pmul(x, y):
    out = np.zeros(np.broadcast_shapes(x.shape[:-1], y.shape[:-1])
                   + (x.shape[-1] + y.shape[-1] - 1,), complex)
    for i in range(x.shape[-1]):
        out[..., i:i + y.shape[-1]] += x[..., i:i + 1] * y
    return out


def _padd(x, y):
    n = max(x.shape[-1], y.shape[-1])
    out = np.zeros(np.broadcast_shapes(x.shape[:-1], y.shape[:-1]) + (n,), complex)
    out[..., :x.shape[-1]] += x
    out[..., :y.shape[-1]] += y
    return out


def _lens_poly(w, e, r):
    """Ascending coefficients of the lens polynomial at lens-frame positions w."""
    nl = len(e)
    col = lambda v: np.broadcast_to(np.asarray(v, complex), w.shape)[..., None]  # noqa: E731
    lin = [np.concatenate([-col(x), np.ones_like(col(x))], -1) for x in r]
    D, N = lin[0], 0
    for j in range(1, nl):
        D = _pmul(D, lin[j])
    terms = []
    for j in range(nl):
        t = col(e[j])
        for k in range(nl):
            if k != j:
                t = _pmul(t, lin[k])
        terms.append(t)
    N = sum(terms)
    M = [_padd((np.conj(w)[..., None] - np.conj(col(x))) * D, N) for x in r]
    prod = M[0]
    for j in range(1, nl):
        prod = _pmul(prod, M[j])
    P = _pmul(np.concatenate([-w[..., None], np.ones_like(w[..., None])], -1), prod)
    S = 0
    for j in range(nl):
        t = col(e[j])
        for k in range(nl):
            if k != j:
                t = _pmul(t, M[k])
        S = S + t
    return _padd(P, -_pmul(D, S))


def _eig_roots(c):
    """Roots of ascending coefficients c (N, n+1) from the companion matrices, two Newton
    steps each."""
    n = c.shape[-1] - 1
    m = np.zeros(c.shape[:-1] + (n, n), complex)
    m[..., 0, :] = -c[..., n - 1::-1] / c[..., n:]
    m[..., np.arange(1, n), np.arange(n - 1)] = 1.0
    z = np.linalg.eigvals(m)
    for _ in range(2):
        p, d = np.broadcast_to(c[..., n:], z.shape), np.zeros_like(z)
        for k in range(n - 1, -1, -1):
            d = d * z + p
            p = p * z + c[..., k:k + 1]
        step = p / d
        z = z - np.where(np.isfinite(step), step, 0)
    return z


def _caustic_points(g, p, nl):
    """One random caustic point per lens, in the frame of the API."""
    e, r, x_cm = _frame(p, nl)
    n = len(p["s"])
    lin2 = []
    for x in r:
        lin = np.stack([-np.asarray(x, complex), np.ones(n, complex)], -1)
        lin2.append(_pmul(lin, lin))
    full, rest = np.exp(1j * g.uniform(0, 2 * np.pi, n))[:, None].astype(complex), 0
    for f in lin2:
        full = _pmul(full, f)
    for j in range(nl):
        t = np.asarray(e[j], complex)[:, None]
        for k in range(nl):
            if k != j:
                t = _pmul(t, lin2[k])
        rest = rest + t
    z = _eig_roots(_padd(full, -rest))
    z = z[np.arange(n), g.integers(0, z.shape[1], n)]
    w = z - sum(e[j] / (np.conj(z) - np.conj(r[j])) for j in range(nl))
    return w - x_cm


def _trajectory(t, t0, u0, tE, alpha):
    tau = (t[None, :] - t0[:, None]) / tE[:, None]
    return (u0[:, None] + 1j * tau) * np.exp(-1j * alpha)[:, None]


def _crossings(g, nl, sets, epochs, npts):
    """Light curves through a caustic point at t = 0 (tE = 20 d, t in [-2 tE, 2 tE]) with
    uneven limb resolutions: npts at the crossing, halved per doubling of the distance in
    source radii down to 256 (npts itself below 256 or for single epochs)."""
    p = _lenses(g, sets, nl)
    rho = _loguniform(g, 1e-3, 3e-2, sets)
    c = _caustic_points(g, p, nl)
    alpha = g.uniform(0, 2 * np.pi, sets)
    rot = c * np.exp(1j * alpha)
    tE = np.full(sets, 20.0)
    if epochs == 1:
        t = np.array([1.5 * 20.0]) * rho[0]
    else:
        t = np.linspace(-40.0, 40.0, epochs)
    w = _trajectory(t, -rot.imag * tE, rot.real, tE, alpha)
    if npts >= 1024:
        x = np.abs(t)[None, :] / 20.0 / rho[:, None]
        k = np.clip(np.ceil(np.log2(np.maximum(x, 1e-300))), 0, None)
        npts = np.clip(npts / 2.0 ** k, 256, npts).astype(np.int32).reshape(-1)
    rep = lambda v: np.repeat(v, t.size)  # noqa: E731
    return w.reshape(-1), rep(rho), {k: rep(v) for k, v in p.items()}, npts


def _gpu(x, grad=False):
    return torch.as_tensor(np.ascontiguousarray(x), device=DEV).requires_grad_(grad)


def _earth(t_jpl):
    """A circular Earth orbit of 1 AU, inclined by the obliquity of the ecliptic."""
    ph, om, ob = 2 * np.pi * t_jpl / 365.25, 2 * np.pi / 365.25, np.deg2rad(23.44)
    pos = np.stack([np.cos(ph), np.sin(ph) * np.cos(ob), np.sin(ph) * np.sin(ob)], -1)
    vel = om * np.stack([-np.sin(ph), np.cos(ph) * np.cos(ob), np.cos(ph) * np.sin(ob)], -1)
    return pos, vel


def _host(case, seed):
    """Host arrays of a case's inputs, made from the seed alone."""
    g = np.random.Generator(np.random.PCG64(np.random.SeedSequence([seed, 7])))
    kind = case["kind"]
    if kind == "curves":
        return dict(_lenses(g, 1, case["nl"]))
    if kind == "ps":
        p = _lenses(g, 1, case["nl"])
        return dict(w=_disk(g, case["n"]), p=p, g=g.normal(size=case["n"]))
    if kind == "lc":
        n = case["l"]
        p = dict(t0=g.uniform(-10, 10, n), u0=g.uniform(-0.5, 0.5, n),
                 tE=_loguniform(g, 5.0, 100.0, n), alpha=g.uniform(0, 2 * np.pi, n),
                 **_lenses(g, n, case["nl"]))
        return dict(t=np.linspace(-60.0, 60.0, case["t"]), p=p, g=g.normal(size=(n, case["t"])))
    if kind == "roots":
        n, nl = case["n"], case["nl"]
        p = _lenses(g, n, nl)
        e, r, x_cm = _frame(p, nl)
        c = _lens_poly(_disk(g, n) + x_cm, e, r)
        d = DEGREE[nl]
        return dict(c=c, g=g.normal(size=(n, d)) + 1j * g.normal(size=(n, d)))
    if kind == "ext":
        w, rho, p, npts = _crossings(g, case["nl"], case["sets"], case["epochs"], case["npts"])
        return dict(w=w, rho=rho, p=p, npts=npts, u1=np.full(w.size, 0.4),
                    g=g.normal(size=w.size))
    if kind == "mag":
        n = case["n"]
        if not case["ragged"]:   # one event: a light curve that passes the caustic
            w, rho, p, _ = _crossings(g, 2, 1, n, 200)
            return dict(w=w, rho=rho, p=p, npts=case["npts_max"], u1=np.full(n, 0.5),
                        g=g.normal(size=n))
        p = _lenses(g, n, 2)
        rho = _loguniform(g, 1e-3, 1e-1, n)
        near = _caustic_points(g, p, 2) + (g.uniform(0, 2, n) * rho
                                           * np.exp(1j * g.uniform(-np.pi, np.pi, n)))
        w = np.where(np.arange(n) < n // 2, near, _disk(g, n))
        sizes = [m for m in (256, 512, 1024, 2048, 4096) if m <= case["npts_max"]]
        return dict(w=w, rho=rho, p=p, npts=g.choice(np.asarray(sizes), n), u1=np.full(n, 0.5),
                    g=g.normal(size=n))
    # infer
    n, T = case["l"], case["t"]
    t = np.sort(g.uniform(8000.0, 8200.0, T))
    q = {"t0": g.uniform(8090, 8110, n), "u0": g.uniform(0.05, 0.5, n),
         "tE": _loguniform(g, 20.0, 60.0, n), "piEE": g.normal(0, 0.2, n),
         "piEN": g.normal(0, 0.2, n), **_lenses(g, n, 2)}
    u = np.hypot(0.2, (t - 8100.0) / 30.0)
    a = (u**2 + 2) / (u * np.sqrt(u**2 + 4))
    err = 0.02 * np.sqrt(a)
    return dict(t=t, p=q, fobs=1.3 * a + 0.4 + err * g.normal(size=T), c_inv=1 / err**2,
                cut=(3 * T) // 5)


def prepare(case, seed):
    h = _host(case, seed)
    kind = case["kind"]
    st = dict(case=case)
    if kind == "curves":
        st["p"] = {k: float(v[0]) for k, v in h.items()}
        return st
    if kind == "ps":
        st["w"] = _gpu(h["w"], case["grad"])
        st["p"] = {k: _gpu(v[0], case["grad"]) for k, v in h["p"].items()}
        st["g"] = _gpu(h["g"])
    elif kind == "lc":
        st["t"] = _gpu(h["t"])
        st["p"] = {k: _gpu(v, True) for k, v in h["p"].items()}
        st["g"] = _gpu(h["g"])
    elif kind == "roots":
        # poly_roots takes the highest power first, ehrlich_aberth the lowest
        c = h["c"][:, ::-1] if case["init"] == "reference" else h["c"]
        st["c"] = _gpu(c, case["grad"])
        st["g"] = _gpu(h["g"])
    elif kind in ("ext", "mag"):
        st["w"], st["rho"] = _gpu(h["w"], case["grad"]), _gpu(h["rho"], case["grad"])
        st["p"] = {k: _gpu(v, case["grad"]) for k, v in h["p"].items()}
        st["u1"], st["npts"], st["g"] = _gpu(h["u1"]), h["npts"], _gpu(h["g"])
    else:
        t_jpl = np.arange(h["t"][0], h["t"][-1] + 1, 1)
        st["traj"] = ca.AnnualParallaxTrajectory(h["t"], (265.0, -28.0), *_earth(t_jpl))
        st["t"] = _gpu(h["t"])
        st["p"] = {k: _gpu(v, True) for k, v in h["p"].items()}
        cut = h["cut"]
        st["fobs"] = [_gpu(h["fobs"][:cut]), _gpu(h["fobs"][cut:])]
        st["c_inv"] = [_gpu(h["c_inv"][:cut]), _gpu(h["c_inv"][cut:])]
        st["cut"] = cut
    return st


def run(st):
    case, kind = st["case"], st["case"]["kind"]
    if kind == "curves":
        return list(ca.critical_and_caustic_curves(npts=case["npts"], nlenses=case["nl"],
                                                   **st["p"]))
    p = st["p"] if kind != "roots" else None
    if kind == "ps":
        m = ca.mag_point_source(st["w"], nlenses=case["nl"], **p)
        if not case["grad"]:
            return [m]
        return [m.detach(), *torch.autograd.grad(m, [st["w"], *p.values()], st["g"])]
    if kind == "lc":
        m = ca.mag_point_source_lightcurve(st["t"], nlenses=case["nl"], **p)
        return [m.detach(), *torch.autograd.grad(m, list(p.values()), st["g"])]
    if kind == "roots":
        if case["init"] == "reference":
            z = ca.poly_roots(st["c"])
        else:
            z = ca.ehrlich_aberth(st["c"], init="complex").reshape(st["g"].shape)
        if not case["grad"]:
            return [z]
        return [z.detach(), *torch.autograd.grad(z, [st["c"]], st["g"])]
    if kind in ("ext", "mag"):
        if kind == "ext":
            m = ca.mag_extended_source(st["w"], st["rho"], nlenses=case["nl"],
                                       npts_limb=st["npts"], limb_darkening=case["ld"],
                                       u1=st["u1"], **p)
        else:
            m = ca.mag(st["w"], st["rho"], nlenses=2, npts_limb=st["npts"], limb_darkening=True,
                       u1=st["u1"], **p)
        if not case["grad"]:
            return [m]
        leaves = [st["w"], st["rho"], *p.values()]
        return [m.detach(), *torch.autograd.grad(m, leaves, st["g"])]
    geo = {k: p[k] for k in ("t0", "u0", "tE", "piEE", "piEN")}
    w = st["traj"].compute(st["t"], **geo)
    m = ca.mag_point_source(w, nlenses=2, s=p["s"][:, None], q=p["q"][:, None])
    cut = st["cut"]
    beta, ll = ca.marginalized_log_likelihood([m[:, :cut], m[:, cut:]], st["fobs"], st["c_inv"])
    return [w.detach(), m.detach(), *[b.detach() for b in beta], ll.detach(),
            *torch.autograd.grad(ll.sum(), list(p.values()))]


# ---- work a pass cannot do without -------------------------------------------------------
# One root needs some 6 Newton-type iterations from a cold start, 28 n + 20 flops each for
# degree n (value, derivative, correction); a contour point 3 from its neighbour.
def _root_flops(n, iters):
    return n * iters * (28 * n + 20)


def work(case):
    kind = case["kind"]
    if kind == "curves":
        n = 4 if case["nl"] == 2 else 6
        return dict(bytes=2 * 16 * n * case["npts"], flops=case["npts"] * _root_flops(n, 6))
    nl = case.get("nl", 2)
    d = DEGREE[nl]
    per_point = _root_flops(d, 6) + (300 if nl == 2 else 1100) + 80 * d
    if kind == "ps":
        n = case["n"]
        extra = 50 * d * (2 + len(LENS_NAMES[nl])) if case["grad"] else 0
        return dict(bytes=n * (16 + 8 + (8 + 16 if case["grad"] else 0)),
                    flops=n * (per_point + extra))
    if kind == "lc":
        n = case["l"] * case["t"]
        return dict(bytes=16 * n, flops=n * (per_point + 50 * d * 6))
    if kind == "roots":
        n = case["n"]
        return dict(bytes=n * 16 * (2 * d + 1) + (n * 16 * (2 * d + 1) if case["grad"] else 0),
                    flops=n * _root_flops(d, 6))
    if kind in ("ext", "mag"):
        if kind == "ext":
            s = case["sets"] * case["epochs"]
            pts = s * (256 if case["npts"] >= 1024 else case["npts"])
        else:
            s = case["n"] if not case["ragged"] else case["n"] // 2
            pts = s * (case["npts_max"] if not case["ragged"] else 1000) // 2
        images = 6 if nl == 3 else 4
        node = (177 if case["grad"] else 62) if case.get("ld", True) else 1
        lines = 200 if case.get("ld", True) else 10
        return dict(bytes=s * 8 * (6 + len(LENS_NAMES[nl]) + (6 if case["grad"] else 0)),
                    flops=pts * (_root_flops(d, 3) + images * lines * node))
    n = case["l"] * case["t"]
    return dict(bytes=16 * n * 5, flops=n * (2 * per_point + 50 * d * 4))


# ---- the same outputs in plain 64-bit numpy / torch -----------------------------------------
def _exact_mag(w, p, nl):
    """Point-source magnification as a differentiable torch (CPU) function of w and the
    lens parameters p: images from the companion matrices, one Newton step of the lens
    equation around them carries the implicit derivative."""
    e, r, x_cm = _frame(p, nl, torch)
    wl = w + x_cm
    shape = wl.shape
    num = lambda v: np.broadcast_to(v.detach().numpy(), shape).reshape(-1)  # noqa: E731
    en, rn, wn = [num(v) for v in e], [num(v) for v in r], num(wl)
    z = np.concatenate([_eig_roots(_lens_poly(wn[i:i + 65536], [v[i:i + 65536] for v in en],
                                              [v[i:i + 65536] for v in rn]))
                        for i in range(0, wn.size, 65536)])
    d = [np.conj(z) - np.conj(x)[:, None] for x in rn]
    G = sum(m[:, None] / v for m, v in zip(en, d))
    K = sum(m[:, None] / v**2 for m, v in zip(en, d))
    real = np.abs(z - G - wn[:, None]) < 1e-6
    zt = torch.as_tensor(z.reshape(*shape, -1))
    Kt = torch.as_tensor(K.reshape(*shape, -1))
    up = lambda v: v.expand(shape)[..., None]  # noqa: E731

    def lens(zz):
        return sum(up(m) / (torch.conj(zz) - torch.conj(up(x))) for m, x in zip(e, r))

    u = up(wl) - (zt - lens(zt))            # residual at the fixed images
    det0 = 1 - Kt.abs() ** 2
    zz = zt + (u - Kt * torch.conj(u)) / det0
    Kd = sum(up(m) / (torch.conj(zz) - torch.conj(up(x))) ** 2 for m, x in zip(e, r))
    # |1 - |K|^2|^-1 over the real images
    det = 1 - (Kd.real**2 + Kd.imag**2)
    ok = torch.as_tensor(real.reshape(*shape, -1))
    return torch.where(ok, 1 / torch.where(ok, det, torch.ones_like(det)).abs(),
                       torch.zeros_like(det)).sum(-1)


def _leaf(x):
    return torch.as_tensor(np.ascontiguousarray(x)).requires_grad_(True)


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("ps", "lc", "infer"):
        return None   # roots come in the solver's order, contours follow its limb points
    h = _host(case, seed)
    if kind == "ps":
        w, p = _leaf(h["w"]), {k: _leaf(v[0]) for k, v in h["p"].items()}
        m = _exact_mag(w, p, case["nl"])
        if not case["grad"]:
            return [m.detach()]
        return [m.detach(), *torch.autograd.grad(m, [w, *p.values()], torch.as_tensor(h["g"]))]
    p = {k: _leaf(v) for k, v in h["p"].items()}
    lens = {k: p[k][:, None] for k in ("s", "q")}
    if kind == "lc":
        t = torch.as_tensor(h["t"])
        tau = (t[None, :] - p["t0"][:, None]) / p["tE"][:, None]
        w = torch.exp(-1j * p["alpha"])[:, None] * torch.complex(
            p["u0"][:, None].expand_as(tau), tau)
        m = _exact_mag(w, lens, 2)
        return [m.detach(), *torch.autograd.grad(m, list(p.values()), torch.as_tensor(h["g"]))]
    # trajectory: the Sun's position interpolated on the daily grid
    t = torch.as_tensor(h["t"])
    t_jpl = np.arange(h["t"][0], h["t"][-1] + 1, 1)
    pos, vel = _earth(t_jpl)
    ra, dec = np.deg2rad([265.0, -28.0])
    d = np.array([np.cos(dec) * np.cos(ra), np.cos(dec) * np.sin(ra), np.sin(dec)])
    east = np.cross([0.0, 0.0, 1.0], d)
    north = np.cross(d, east)
    east, north = east / np.linalg.norm(east), north / np.linalg.norm(north)
    grid = torch.as_tensor(t_jpl)

    def at(tab, x):
        tab = torch.as_tensor(np.ascontiguousarray(tab))
        i = (torch.searchsorted(grid, x.detach(), right=True)).clamp(1, grid.numel() - 1)
        y = tab[i - 1] + (x - grid[i - 1]) / (grid[i] - grid[i - 1]) * (tab[i] - tab[i - 1])
        y = torch.where(x.detach() < grid[0], tab[0], y)
        return torch.where(x.detach() > grid[-1], tab[-1], y)

    piE = torch.sqrt(p["piEE"] ** 2 + p["piEN"] ** 2)
    psi = torch.atan2(p["piEE"], p["piEN"])
    dt = t[None, :] - p["t0"][:, None]
    ds = []
    for axis in (east, north):
        ds.append(at(-pos @ axis, t)[None, :] - at(-pos @ axis, p["t0"])[:, None]
                  - dt * at(-vel @ axis, p["t0"])[:, None])
    tau, u0 = dt / p["tE"][:, None], p["u0"][:, None]
    cs, sn, pe = torch.cos(psi)[:, None], torch.sin(psi)[:, None], piE[:, None]
    w = torch.complex(u0 * cs + tau * sn + pe * ds[0], -u0 * sn + tau * cs + pe * ds[1])
    m = _exact_mag(w, lens, 2)
    ll, beta = 0, []
    for sl in (slice(0, h["cut"]), slice(h["cut"], None)):
        A, f, c = m[:, sl], torch.as_tensor(h["fobs"][sl]), torch.as_tensor(h["c_inv"][sl])
        X = torch.stack([A, torch.ones_like(A)], -1)
        N = X.transpose(1, 2) @ (c[None, :, None] * X)
        b = torch.linalg.solve(N, (X * (c * f)[None, :, None]).sum(1))
        res = f - (X @ b[:, :, None])[..., 0]
        chi2 = (c * res**2).sum(-1)
        ll = ll - 0.5 * chi2 + 0.5 * (2 * math.log(2 * math.pi) - torch.logdet(N))
        beta.append(b.detach())
    return [w.detach(), m.detach(), *beta, ll.detach(),
            *torch.autograd.grad(ll.sum(), list(p.values()))]
