"""Contour results of a source by itself and of the same source in a large batch, which other
kernels solve (small batches: groups of lanes)."""
import numpy as np
import pytest
import torch

import caustics_amd as ca
from caustics_amd import _lib
from caustics_amd.extended_source import _run

pytestmark = pytest.mark.gpu

LENSES = {
    "binary": dict(s=0.9, q=0.4),
    "planet": dict(s=0.7, q=1e-5),
    "triple": dict(s=0.9, q=0.4, q3=0.3, r3=0.8, psi=0.7),
    "triple_planet": dict(s=1.1, q=1e-3, q3=1e-6, r3=1.2, psi=2.1),
}


def at_caustics(lens, rho, S, seed=1):
    """S source centres within two radii of the lens' caustics."""
    r = np.random.default_rng(seed)
    nl = 2 if len(LENSES[lens]) == 2 else 3
    c = ca.critical_and_caustic_curves(npts=400, nlenses=nl, **LENSES[lens])[1]
    return nl, r.choice(c.reshape(-1).cpu().numpy(), S) + \
        rho * r.uniform(0, 2, S) * np.exp(2j * np.pi * r.uniform(size=S))


def alone_and_among(lens, rho, S, itmax=2500, npts=200, ld=False):
    """(mag, status, gradients) of S sources as a call of their own and among skipped ones,
    which make the call large."""
    nl, w = at_caustics(lens, rho, S)
    f64 = lambda x: torch.as_tensor(x, dtype=torch.float64, device="cuda")  # noqa: E731
    out = []
    for pad in (0, 1300):
        n = S + pad
        prm = f64([list(LENSES[lens].values())]).expand(n, -1).contiguous()
        wt = torch.as_tensor(np.resize(w, n), device="cuda")
        res = _run(nl, wt, f64(np.full(n, rho)), prm, None, npts, ld,
                   f64(np.full(n, 0.4)) if ld else None, 20, itmax, _lib.MODE_FP64,
                   g=f64(np.ones(n)), skip=torch.arange(n, device="cuda") >= S)
        out.append([x[:S].cpu().numpy() for x in res])
    return out


@pytest.mark.parametrize("lens", list(LENSES))
@pytest.mark.parametrize("itmax", [1, 5, 8, 12, 16, 20, 249])
def test_iteration_limit_means_the_same_in_every_batch(gpu, lens, itmax):
    """A limit on the sweeps stops the same solves whatever else is in the call."""
    alone, among = alone_and_among(lens, 1e-3, 60, itmax)
    for a, b in zip(alone, among):
        np.testing.assert_array_equal(a, b)
    assert itmax < 249 or alone[1].all()
    assert itmax > 8 or not alone[1].all()


@pytest.mark.parametrize("ld", [False, True])
@pytest.mark.parametrize("rho", [1e-2, 1e-3, 1e-4])
@pytest.mark.parametrize("lens", list(LENSES))
def test_sources_at_caustics_by_themselves_and_in_a_large_call(gpu, lens, rho, ld):
    """At caustics, with third lenses down to 1e-6, where an ulp in a coefficient moves roots by
    1e-6 and magnifications by per cent: both ways have to round the coefficients alike and
    polish the roots to the same doubles.  Only roots of a nearly double pair that has not come
    to rest may differ: an ulp of such an image, 2e-16, is magnified by 1/|det J|, at most some
    1e4 at these distances, once into the magnification's integrand and twice into a
    derivative's."""
    alone, among = alone_and_among(lens, rho, 300, ld=ld)
    np.testing.assert_array_equal(alone[1], among[1])
    np.testing.assert_allclose(alone[0], among[0], rtol=1e-11, atol=0.0)
    largest = np.abs(among[2]).max(1, keepdims=True)
    assert (np.abs(alone[2] - among[2]) <= 1e-8 * largest).all()


# few sources: groups of lanes, cut line integrals; many: the flat kernels; limb sizes of both
# selection kernels (512 points are one wave's)
@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("npts", [512, 1024])
@pytest.mark.parametrize("S", [6, 1300])
@pytest.mark.parametrize("lens", ["binary", "triple"])
def test_workspace_contents_do_not_change_results(gpu, lens, S, npts, grad):
    """Every workspace read is of memory that the same launch sequence wrote before, on every
    route: a workspace holding the 64-bit value 1 in every word gives the bits of a zero-filled
    one (a stale index would read 0 or 1 there, a stale double a tiny number)."""
    from caustics_amd.extended_source import extended_workspace_bytes

    rho = 1e-2
    nl, w = at_caustics(lens, rho, S)
    g = np.random.default_rng(S)
    sizes = g.choice([4, 20, npts // 2, npts], S).astype(np.int32)
    sizes[:2] = npts, 0   # one of the largest, one skipped
    dev = lambda x: torch.as_tensor(x, device="cuda").contiguous()  # noqa: E731
    wt, rho_t, u1 = dev(w), dev(np.full(S, rho)), dev(np.full(S, 0.4))
    prm = dev(np.tile(list(LENSES[lens].values()), (S, 1)))
    nt, gm = dev(sizes), dev(g.normal(size=S)) if grad else None
    nb = extended_workspace_bytes(nl, S, npts)
    out = []
    for fill in (0, 1):
        ws = torch.full(((nb + 7) // 8,), fill, dtype=torch.int64, device="cuda")
        mag = torch.empty(S, dtype=torch.float64, device="cuda")
        st = torch.empty(S, dtype=torch.uint8, device="cuda")
        go = torch.zeros((S, 4 + prm.shape[1]), dtype=torch.float64, device="cuda")
        _lib.check(_lib.lib().caus_mag_extended_source_work(
            _lib.stream_ptr(), nl, _lib.ptr(wt), S, _lib.ptr(rho_t), _lib.ptr(prm), prm.shape[1],
            _lib.ptr(nt), npts, 1, _lib.ptr(u1), 1, 20, _lib.ptr(gm), _lib.ptr(mag),
            _lib.ptr(go) if grad else None, _lib.ptr(st), _lib.ptr(ws), ws.numel() * 8, 2500,
            _lib.MODE_FP64, None), "caus_mag_extended_source_work")
        torch.cuda.synchronize()
        out.append((mag, go, st))
    for a, b in zip(*out):
        assert torch.equal(a, b)
    assert out[0][0][1].item() == 0 and bool(torch.isfinite(out[0][0]).all())
