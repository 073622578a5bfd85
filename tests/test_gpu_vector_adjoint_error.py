"""Error of the adjoint of the vector synthesis against its definition in long double, for
orders 0, 1 and 2 of noise on Gauss grids.  sin(theta) dP_l/dtheta is l x P_l - g_l P_{l-1}, two terms
of the size l P_l each, so with values good to eps a sum of them is good to about lmax eps;
the bound is twice that."""
import numpy as np
import pytest

from _util import to_dev, to_host

pytestmark = pytest.mark.gpu

LD = np.longdouble
PI = LD("3.14159265358979323846264338327950288")


def _legendre(m, lmax, x):
    """P_l^m (orthonormal, no Condon-Shortley phase), l = m .. lmax, in long double."""
    s = np.sqrt((1 - x) * (1 + x))
    P = np.zeros((lmax + 1 - m, x.size), LD)
    P[0] = 1 / np.sqrt(4 * PI)
    for k in range(1, m + 1):
        P[0] *= np.sqrt(LD(2 * k + 1) / LD(2 * k)) * s
    a = lambda l: np.sqrt(LD(4 * l * l - 1) / LD(l * l - m * m))
    for l in range(m + 1, lmax + 1):
        P[l - m] = a(l) * (x * P[l - 1 - m] - (P[l - 2 - m] / a(l - 1) if l - 2 >= m else 0))
    return P


def _derivative(m, lmax, x):
    """dP_l^m/dtheta; order 0 from order 1 (no cancellation)."""
    D = np.zeros((lmax + 1 - m, x.size), LD)
    if m == 0:
        l = np.arange(1, lmax + 1).astype(LD)
        D[1:] = -np.sqrt(l * (l + 1))[:, None] * _legendre(1, lmax, x)
        return D
    s, P = np.sqrt((1 - x) * (1 + x)), _legendre(m, lmax, x)
    for l in range(m, lmax + 1):
        D[l - m] = l * x * P[l - m]
        if l > m:
            D[l - m] -= np.sqrt(LD((2 * l + 1) * (l * l - m * m)) / LD(2 * l - 1)) * P[l - 1 - m]
        D[l - m] /= s
    return D


def _error(got, ref):
    """Relative L2 distance up to one real factor (normalisation and phase)."""
    c = (np.vdot(ref, got) / np.vdot(ref, ref)).real
    return float(np.linalg.norm(got - c * ref) / np.linalg.norm(c * ref))


@pytest.mark.parametrize("lmax,nlat,nlon,nf", [
    (255, 256, 512, 1),
    (255, 256, 512, 4),
])
def test_error_of_low_orders(shtk, cuda, lmax, nlat, nlon, nf):
    cfg = shtk.create_gauss_config(lmax, nlat, nlon=nlon)
    rng = np.random.default_rng(7)
    V = [np.asfortranarray(rng.standard_normal((nlat, nlon, nf))) for _ in range(2)]
    print(f"adjoint lmax={lmax} nf={nf}", flush=True)
    got = [to_host(g).astype(np.clongdouble) for g in shtk._adjoint_synthesis_sphtor(cfg, *[to_dev(v) for v in V])]
    x = cfg.x.astype(LD)
    s = np.sqrt((1 - x) * (1 + x))
    for m in (0, 1, 2):
        P, D = _legendre(m, lmax, x), _derivative(m, lmax, x)
        t = 2 * PI * ((m * np.arange(nlon)) % nlon) / nlon
        e = np.cos(t) - 1j * np.sin(t)
        lo = max(1, m)
        for k in range(nf):
            Ft, Fp = [v[:, :, k].astype(LD) @ e for v in V]
            S = (D @ Ft - 1j * m * (P @ (Fp / s)))[lo - m:]
            T = (1j * m * (P @ (Ft / s)) + D @ Fp)[lo - m:]
            for g, r in zip(got, (S, T)):
                assert _error(g[lo:, m, k], r) < 2 * lmax * 2.0 ** -52, (m, k)
