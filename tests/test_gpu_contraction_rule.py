"""Which contraction a call of each precision runs, by the names of its kernel events, on both
sides of every line of the rule; and syntheses of FP32 arrays by the field groups, which read
them without a conversion pass, against the oracle (values in FP64, so the bound is the
rounding of the FP32 grid, 6e-8, with room for its sums: 1e-6)."""
import numpy as np
import pytest
import torch

from _util import rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu

# few orders: the rule looks at degrees, latitudes, fields and dtype
CASES = [
    # lmax, nlat, nf, dtype, precision, synthesis event, analysis event
    (1000, 2000, 16, "f64", "split", "oz_synth", "leg_anal"),
    (1000, 2000, 15, "f64", "split", "oz_synth", "leg_anal"),
    (1000, 2000, 15, "f32", "split", "oz_synth", "leg_anal"),
    (1000, 2000, 14, "f64", "split", "leg_synth", "leg_anal"),
    (1000, 2000, 28, "f64", "split", "leg_synth", "leg_anal"),
    (1000, 1998, 16, "f64", "split", "leg_synth", "leg_anal"),
    (511, 512, 16, "f32", "fp32", "leg_synth", "leg_anal"),
    (900, 901, 16, "f32", "fp32", "f32_synth", "leg_anal"),
    (900, 901, 24, "f32", "fp32", "leg_synth", "leg_anal"),
    (899, 901, 16, "f32", "fp32", "leg_synth", "leg_anal"),
    (255, 256, 4, "f64", "fp32", "f32_synth", "f32_anal"),
    (255, 256, 16, "f64", "fp64", "leg_synth", "leg_anal"),
]


@pytest.mark.parametrize("lmax,nlat,nf,dtype,precision,synth,anal", CASES)
def test_contraction_that_runs(shtk, oracle, cuda, lmax, nlat, nf, dtype, precision, synth, anal):
    from shtnskit_jl_amd import _lib

    mmax, nlon = 6, 16
    cfg = shtk.create_gauss_config(lmax, nlat, nlon=nlon, mmax=mmax)
    alm = oracle.random_alm(lmax, mmax, seed=nf, power=1.0, nf=nf)
    d = to_dev(alm.astype(np.complex64 if dtype == "f32" else np.complex128))
    print(f"rule lmax={lmax} nlat={nlat} nf={nf} {dtype} {precision}", flush=True)
    _lib.profile_enable(cfg.plan, True)
    f = shtk.synthesis_batch(cfg, d, precision=precision)
    names_s = set(_lib.profile_read(cfg.plan))
    back = shtk.analysis_batch(cfg, f, precision=precision)
    names_a = set(_lib.profile_read(cfg.plan))
    _lib.profile_enable(cfg.plan, False)
    tol = {"f32": 2e-6, "f64": 2e-6 if precision == "fp32" else 1e-11}[dtype]
    ref = to_host(shtk.synthesis_batch(cfg, to_dev(alm)))
    assert max(rel_l2(to_host(f)[..., k], ref[..., k]) for k in range(nf)) < tol
    assert max(rel_l2(to_host(back)[..., k], alm[..., k]) for k in range(nf)) < 2 * tol
    assert names_s == {synth, "fft_synth"} and names_a == {anal, "fft_anal"}


@pytest.mark.parametrize("lmax,nlat,nlon,mres,ltr,nf", [
    (3, 4, 8, 1, -1, 2), (63, 64, 128, 1, -1, 16), (64, 127, 130, 1, 50, 9), (130, 257, 264, 2, -1, 7),
    (255, 256, 512, 1, 201, 12), (300, 302, 640, 1, -1, 48),
])
def test_fp32_arrays_match_oracle(shtk, oracle, cuda, lmax, nlat, nlon, mres, ltr, nf):
    cfg = shtk.create_gauss_config(lmax, nlat, nlon=nlon, mres=mres)
    alm = oracle.random_alm(lmax, lmax, seed=lmax, power=1.0, nf=nf).astype(np.complex64)
    ref = oracle.Config(lmax, nlat, nlon=nlon, mres=mres).synthesis(alm.astype(np.complex128), ltr=ltr)
    if 0 <= ltr < lmax:
        alm[ltr + 1:] = np.nan  # not read
    print(f"FP32 arrays lmax={lmax} nlat={nlat} mres={mres} ltr={ltr} nf={nf}", flush=True)
    for precision in ("fp64", "fp32"):
        got = shtk.synthesis_batch(cfg, to_dev(alm), ltr=ltr, precision=precision)
        assert got.dtype == torch.float32
        assert max(rel_l2(to_host(got)[..., k], ref[..., k]) for k in range(nf)) < 1e-6
