"""Field-group synthesis by one wave per unit, the form of launches with 8192 units or more
(orders x blocks of 64 pairs x groups), over orders of several segments: chains that hand
over from scaled to live inside the unit, seeds loaded a segment ahead, and the vector pair's
edge terms at every segment, for each group size, against the oracle (FP64, 1e-12)."""
import numpy as np
import pytest
import torch

from _util import rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _check(got, ocfg_call, ks):
    """Compares the fields ks of the device grids with the oracle's."""
    refs = ocfg_call(ks)
    for g, r in zip(got, refs):
        for i, k in enumerate(ks):
            assert rel_l2(to_host(g[..., k]), r[..., i]) < TOL, k


@pytest.mark.parametrize("lmax,nlat,nlon,ltr,nf", [
    (1023, 1024, 2048, -1, 2), (1023, 1024, 2048, 990, 3), (1023, 1025, 2048, -1, 4),
    (700, 702, 1440, -1, 10), (700, 702, 1440, 650, 12), (700, 703, 1440, -1, 14), (700, 702, 1440, -1, 16),
    (300, 302, 640, -1, 80),
])
def test_scalar(shtk, oracle, cuda, lmax, nlat, nlon, ltr, nf):
    cfg, ocfg = shtk.create_gauss_config(lmax, nlat, nlon=nlon), oracle.Config(lmax, nlat, nlon=nlon)
    assert (lmax + 1) * (((nlat + 1) // 2 + 63) // 64) * ((nf + 7) // 8) >= 8192
    alm = oracle.random_alm(lmax, lmax, seed=nf, power=1.0, nf=nf)
    print(f"one wave lmax={lmax} nlat={nlat} ltr={ltr} nf={nf}", flush=True)
    for dtype in (np.complex128, np.complex64):
        a = alm.astype(dtype)
        got = shtk.synthesis_batch(cfg, to_dev(a), ltr=ltr)
        if dtype == np.complex128:
            f64 = got
            _check([got], lambda ks: [ocfg.synthesis(np.asfortranarray(a[..., ks]), ltr=ltr)], [0, nf - 1])
        else:  # 6e-8 in the coefficients and in the grid
            assert torch.linalg.vector_norm(got - f64) < 2e-7 * torch.linalg.vector_norm(f64)


@pytest.mark.parametrize("lmax,nlat,nlon,ltr,nf", [
    (1023, 1024, 2048, -1, 1), (1023, 1024, 2048, 895, 2), (700, 702, 1440, -1, 5), (700, 703, 1440, 640, 8),
])
def test_vector(shtk, oracle, cuda, lmax, nlat, nlon, ltr, nf):
    cfg, ocfg = shtk.create_gauss_config(lmax, nlat, nlon=nlon), oracle.Config(lmax, nlat, nlon=nlon)
    assert (lmax + 1) * (((nlat + 1) // 2 + 63) // 64) * ((2 * nf + 7) // 8) >= 8192
    S, T = [oracle.random_alm(lmax, lmax, seed=s, power=2.0, nf=nf, lmin=1) for s in (nf, nf + 1)]
    print(f"one wave, vector lmax={lmax} nlat={nlat} ltr={ltr} nf={nf}", flush=True)
    got = shtk.synthesis_sphtor_batch(cfg, to_dev(S), to_dev(T), ltr=ltr)
    _check(got, lambda ks: ocfg.synthesis_sphtor(np.asfortranarray(S[..., ks]), np.asfortranarray(T[..., ks]), ltr=ltr),
           [0, nf - 1])


def test_vector_adjoints_lmax1023(shtk, oracle, cuda):
    """The adjoint of the synthesis sums unweighted rows, those near the poles divided by
    sin(theta): 2e-12 in the lowest orders, so 1e-11; the adjoint of the analysis is a synthesis."""
    lmax, nlat, nlon = 1023, 1024, 2048
    cfg, ocfg = shtk.create_gauss_config(lmax, nlat, nlon=nlon), oracle.Config(lmax, nlat, nlon=nlon)
    rng = np.random.default_rng(5)
    V = [np.asfortranarray(rng.standard_normal((nlat, nlon))) for _ in range(2)]
    S, T = [oracle.random_alm(lmax, lmax, seed=s, power=2.0, lmin=1) for s in (3, 4)]
    print("vector adjoints lmax=1023", flush=True)
    for g, r in zip(shtk._adjoint_synthesis_sphtor(cfg, *[to_dev(v) for v in V]), ocfg.adjoint_synthesis_sphtor(*V)):
        assert rel_l2(to_host(g), r) < 1e-11
    for g, r in zip(shtk._adjoint_analysis_sphtor(cfg, to_dev(S), to_dev(T)), ocfg.adjoint_analysis_sphtor(S, T)):
        assert rel_l2(to_host(g), r) < TOL
