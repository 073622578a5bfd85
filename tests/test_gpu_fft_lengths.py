"""GPU parity of the longitude transform over its kinds of length, against the FP64
oracle: every prime butterfly alone, first and after another pass (7 takes two
butterflies per thread), the generic pass, Bluestein lengths from the smallest to
the longest convolution, odd and even, with and without the bin nlon / 2.

Tolerance: a transform of length n is off by about eps log2(n) relative to its norm,
under 4e-15 at 8192; Bluestein's two longer ones and the chirps by a few times
that; the repository's 1e-12 leaves a factor of a hundred.
"""
import numpy as np
import pytest

from _util import rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu

TOL = 1e-12

# nlon: kind
LENGTHS = [7, 49, 56, 11, 13, 143, 17, 221, 19, 361, 608, 1001, 23, 46, 667, 61, 67, 134, 131, 499, 1018, 2039, 4093,
           8190, 16, 48, 128, 256, 2048, 4096, 8192]


@pytest.mark.parametrize("nlon", LENGTHS)
def test_longitude_lengths(shtk, oracle, cuda, nlon):
    lmax = min(20, (nlon - 1) // 2)
    nlat = lmax + 3
    nf = 3
    mres = 3 if nlon == 1018 else 1
    cfg = shtk.create_gauss_config(lmax, nlat, nlon=nlon, mres=mres)
    ocfg = oracle.Config(lmax, nlat, nlon=nlon, mres=mres)
    print(f"nlon={nlon} lmax={lmax}", flush=True)
    alm = oracle.random_alm(lmax, lmax, seed=nlon, power=1.0, nf=nf)
    alm[:, np.arange(lmax + 1) % mres != 0] = 0.0
    rng = np.random.default_rng(nlon)
    g = np.asfortranarray(rng.standard_normal((nlat, nlon, nf)))
    assert rel_l2(to_host(shtk.synthesis_batch(cfg, to_dev(alm))), ocfg.synthesis(alm)) < TOL
    assert rel_l2(to_host(shtk.analysis_batch(cfg, to_dev(g))), ocfg.analysis(g)) < TOL
    gc = np.asfortranarray(rng.standard_normal((nlat, nlon)) + 1j * rng.standard_normal((nlat, nlon)))
    a0 = np.asfortranarray(alm[:, :, 0])
    assert rel_l2(to_host(shtk.synthesis(cfg, to_dev(a0), real_output=False)), ocfg.synthesis(a0, real_output=False)) < TOL
    assert rel_l2(to_host(shtk.analysis(cfg, to_dev(gc))), ocfg.analysis_cplx(gc)) < TOL
    f32 = to_host(shtk.synthesis(cfg, to_dev(a0.astype(np.complex64))))
    assert f32.dtype == np.float32 and rel_l2(f32, ocfg.synthesis(a0.astype(np.complex64).astype(np.complex128))) < 1e-6


@pytest.mark.parametrize("lmax,nlon", [(20, 41), (20, 42), (48, 97), (33, 68), (66, 133), (66, 134)])
def test_full_rows(shtk, oracle, cuda, lmax, nlon):
    """nlon = 2 lmax + 1 and 2 lmax + 2: every bin is written, or all but nlon / 2; fields
    of large values first, so that a bin left from another tile would show."""
    nlat = 2 * lmax + 6
    cfg = shtk.create_gauss_config(lmax, nlat, nlon=nlon)
    ocfg = oracle.Config(lmax, nlat, nlon=nlon)
    alm = oracle.random_alm(lmax, lmax, seed=lmax, power=1.0, nf=64)
    alm[:, :, ::2] *= 1e6
    f, ref = to_host(shtk.synthesis_batch(cfg, to_dev(alm))), ocfg.synthesis(alm)
    assert max(rel_l2(f[..., k], ref[..., k]) for k in range(64)) < TOL
