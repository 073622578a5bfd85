"""How batches are dealt to the field-group kernels: the launches of an analysis whose last
group holds one or two fields, and groups of 2, 4 and 8 fields of short syntheses against
the oracle (FP64, the FP64 path's 1e-12 relative L2)."""
import numpy as np
import pytest

from _util import rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu

TOL = 1e-12


@pytest.mark.parametrize("lmax,nf,launches", [
    (63, 8, 1), (63, 9, 1), (127, 10, 1), (255, 17, 1), (399, 9, 1),   # one launch more costs more than it saves
    (400, 9, 2), (599, 18, 1), (600, 18, 2), (600, 11, 1),
])
def test_launches_of_an_analysis(shtk, oracle, cuda, lmax, nf, launches):
    from shtnskit_jl_amd import _lib

    nlat, nlon = lmax + 1, 2 * lmax + 2
    cfg = shtk.create_gauss_config(lmax, nlat, nlon=nlon)
    f = np.asfortranarray(np.random.default_rng(nf).standard_normal((nlat, nlon, nf)))
    print(f"analysis lmax={lmax} nf={nf}", flush=True)
    fd = to_dev(f)
    _lib.profile_enable(cfg.plan, True)
    got = to_host(shtk.analysis_batch(cfg, fd))
    count = _lib.profile_read(cfg.plan)["leg_anal"][1]
    _lib.profile_enable(cfg.plan, False)
    ks = [0, 7, nf - 1]  # first group, its last field, the rest
    ref = oracle.Config(lmax, nlat, nlon=nlon).analysis(np.asfortranarray(f[..., ks]))
    assert max(rel_l2(got[..., k], ref[..., i]) for i, k in enumerate(ks)) < TOL
    assert count == launches


@pytest.mark.parametrize("lmax,nlat,nf", [
    (63, 64, 16), (63, 64, 5),        # groups of 2
    (127, 128, 32), (191, 192, 16),   # of 4
    (255, 256, 16),                   # of 8, at 1024 units
    (254, 256, 16),                   # of 4, one order below
])
def test_short_syntheses_match_oracle(shtk, oracle, cuda, lmax, nlat, nf):
    nlon = 2 * lmax + 2
    cfg, ocfg = shtk.create_gauss_config(lmax, nlat, nlon=nlon), oracle.Config(lmax, nlat, nlon=nlon)
    alm = oracle.random_alm(lmax, lmax, seed=nf, power=1.0, nf=nf)
    S, T = [oracle.random_alm(lmax, lmax, seed=s, power=1.0, nf=nf // 2, lmin=1) for s in (1, 2)]
    print(f"synthesis lmax={lmax} nf={nf}", flush=True)
    got = [shtk.synthesis_batch(cfg, to_dev(alm)), *shtk.synthesis_sphtor_batch(cfg, to_dev(S), to_dev(T))]
    for g, r in zip(got, [ocfg.synthesis(alm), *ocfg.synthesis_sphtor(S, T)]):
        g = to_host(g)
        assert max(rel_l2(g[..., k], r[..., k]) for k in range(r.shape[-1])) < TOL
