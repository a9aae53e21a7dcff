"""caus_match_chain against the greedy rule (reference: match_points,
src/caustics/utils.py:15-40) applied point after point."""
import numpy as np
import pytest
import torch

from caustics_amd import _lib

pytestmark = pytest.mark.gpu


def greedy_chain(p):
    """Rows in order take the nearest unused row of the next point (ties, and distances
    that are no numbers, to the first unused one, as a strict comparison in row order
    leaves them)."""
    out = np.empty_like(p)
    prev = p[0]
    for k in range(len(p)):
        free = list(range(p.shape[1]))
        for i in range(p.shape[1]):
            e = p[k][free] - prev[i]
            d = e.real**2 + e.imag**2
            best = 0
            for u in range(1, len(free)):
                if d[u] < d[best]:
                    best = u
            out[k, i] = p[k, free.pop(best)]
        prev = out[k]
    return out


@pytest.mark.parametrize("n", [2, 4, 5, 6, 10])
@pytest.mark.parametrize("npts", [1, 2, 64, 65, 257, 700])
def test_match_chain_is_the_greedy_rule(gpu, n, npts):
    """Chains of 1 to 11 batches of 64 points: smooth rows in shuffled order, independent
    points (most steps conflict), points on a coarse grid (ties and coincident rows), and
    a smooth chain with values that are not finite.  The output holds the input's values,
    so it is compared exactly."""
    g = np.random.default_rng(100 * n + npts)
    t = np.linspace(0, 2 * np.pi, npts)[:, None]
    smooth = np.exp(1j * t * (1 + np.arange(n))) * (1 + np.arange(n))
    smooth = np.take_along_axis(smooth, g.permuted(np.tile(np.arange(n), (npts, 1)), axis=1), 1)
    wild = g.normal(size=(npts, n)) + 1j * g.normal(size=(npts, n))
    grid = g.integers(-2, 3, (npts, n)) + 1j * g.integers(-2, 3, (npts, n))
    odd = smooth.copy()
    odd[npts // 2, n // 2] = np.nan
    odd[npts // 3, 0] = complex(np.inf, 0.0)
    x = np.stack([smooth, wild, grid.astype(complex), odd])
    p = torch.as_tensor(x, device="cuda")
    o = torch.full_like(p, -7.0)
    rc = _lib.lib().caus_match_chain(_lib.stream_ptr(), _lib.ptr(p), _lib.ptr(o), npts, n, len(x))
    _lib.check(rc, "caus_match_chain")
    for c in range(len(x)):
        with np.errstate(invalid="ignore"):
            ref = greedy_chain(x[c])
        np.testing.assert_array_equal(o[c].cpu().numpy(), ref)


@pytest.mark.parametrize("n", [2, 4, 5, 6, 10])
@pytest.mark.parametrize("npts", [1, 2, 12, 13])
def test_many_short_chains(gpu, n, npts):
    """16,384 chains and one more, of up to 12 points (a lane each) and of 13, equal the same
    chains a few at a time."""
    g = np.random.default_rng(10 * n + npts)
    few = g.normal(size=(511, npts, n)) + 1j * g.normal(size=(511, npts, n))
    few[::7] = g.integers(-2, 3, few[::7].shape)          # ties and coincident rows
    few[3, npts // 2, n // 2] = np.nan
    few[5, npts // 3, 0] = complex(np.inf, 0.0)
    many = np.resize(few, (16385, npts, n))

    def chain(x):
        p = torch.as_tensor(x, device="cuda")
        o = torch.full_like(p, -7.0)
        _lib.check(_lib.lib().caus_match_chain(_lib.stream_ptr(), _lib.ptr(p), _lib.ptr(o), npts,
                                               n, len(x)), "caus_match_chain")
        return o.cpu().numpy()

    np.testing.assert_array_equal(chain(many), np.resize(chain(few), many.shape))
