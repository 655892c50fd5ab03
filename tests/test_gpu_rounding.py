"""Rounding that does not average out: an error in a launch constant is the same
in every element, so the energy x.Kx shows it where a norm of K x - y does not."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LD = np.longdouble


def _stiffness(x, n, h):
    """sum over the elements of the Q1 stiffness, in extended precision; x: (nz, ny, nx)"""
    def d(a, ax):
        g = np.diff(a, axis=ax)
        pad = [(0, 0)] * 3
        pad[ax] = (1, 0)
        lo = np.pad(g, pad)
        pad[ax] = (0, 1)
        return (lo - np.pad(g, pad)) / h[ax]

    def m(a, ax):
        a = np.moveaxis(a, ax, 0)
        y = np.zeros_like(a)
        y[:-1] += 2 * a[:-1] + a[1:]
        y[1:] += 2 * a[1:] + a[:-1]
        return np.moveaxis(y, 0, ax) * (h[ax] / LD(6))

    return m(m(d(x, 2), 1), 0) + m(m(d(x, 1), 2), 0) + m(m(d(x, 0), 2), 1)


@pytest.mark.parametrize("n,l", [((24, 10, 31), (1.7, 1.2, 1.7)), ((14, 30, 28), (1.0, 1.6, 0.9)), ((17, 17, 17), (1.0, 1.0, 1.0))],
                         ids=lambda v: "x".join(map(str, v)))
def test_v_stiffness_constants(n, l):
    # AT1 without strain: K is the stiffness alone.  A constant rounded once is
    # off by 1.11e-16 at most, and so is the energy, a mean over the modes of
    # one sign; the products' own rounding averages to 1e-16 / sqrt(nodes)
    import vpfhf_amd as V
    eps = 2 * l[0] / (n[0] - 1)
    P = V.Problem(n, l, nu=0.2, eta=1e-5, epsilon=eps, atnum=1)
    P.set_fields(V=np.ones(P.nn), VIrrev=np.ones(P.nn))
    P.VIJacobian_setup(np.zeros(3 * P.nn))
    x = np.random.default_rng(1).standard_normal(P.nn)
    y = P.VIJacobian_mult(x).astype(LD)
    P.close()
    h = [LD(np.float64(l[d]) / np.float64(n[d] - 1)) for d in (2, 1, 0)]
    c = LD(0.5) / LD(np.float64(2.0) / 3.0) * LD(np.float64(eps))
    ref = c * _stiffness(x.astype(LD).reshape(n[::-1]), n, h).ravel()
    shift = float((x * (y - ref)).sum() / (x * ref).sum())
    assert abs(shift) <= 1.2e-16, shift
