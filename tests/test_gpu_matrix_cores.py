"""The matrix-core contractions where calls still run them, told by the names of their kernel
events: split and FP32 syntheses of many degrees and pairs (few orders, so that the oracle
stays quick) with truncation, orders between multiples of mres, conventions, complex64
coefficients and complex grids, the grouped split synthesis of uneven batches, and every
split and FP32 kernel of both directions on plans with 128-degree segments.  Bounds: the
split path's 1e-11 relative L2 per field, the FP32 path's 2e-6."""
import ctypes

import numpy as np
import pytest
import torch

from _util import rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu

TOL = {"split": 1e-11, "fp32": 2e-6}
EVENT = {"split": "oz", "fp32": "f32"}


def _worst(got, ref):
    got = to_host(got)
    return max(rel_l2(got[..., k], ref[..., k]) for k in range(ref.shape[-1]))


def _traced(plan, call):
    """The call's result and the names of its kernel events."""
    from shtnskit_jl_amd import _lib

    _lib.profile_enable(plan, True)
    out = call()
    names = set(_lib.profile_read(plan))
    _lib.profile_enable(plan, False)
    return out, names


LARGE = [
    # precision, lmax, nlat, nlon, mmax, mres, ltr, nf, conventions
    ("split", 1000, 2000, 64, 20, 1, -1, 15, {}),
    ("split", 1000, 2000, 64, 20, 2, 777, 16, {}),
    ("split", 1023, 2001, 48, 15, 1, 960, 31, dict(norm="schmidt", cs_phase=False, real_norm=True)),
    ("fp32", 900, 901, 64, 20, 1, -1, 16, {}),
    ("fp32", 927, 930, 64, 21, 3, 800, 15, {}),
    ("fp32", 959, 1300, 48, 15, 1, -1, 32, dict(norm="schmidt", cs_phase=False, real_norm=True)),
]


@pytest.mark.parametrize("precision,lmax,nlat,nlon,mmax,mres,ltr,nf,conv", LARGE)
def test_large_syntheses(shtk, oracle, cuda, precision, lmax, nlat, nlon, mmax, mres, ltr, nf, conv):
    kw = dict(nlon=nlon, mmax=mmax, mres=mres, **conv)
    cfg, ocfg = shtk.create_gauss_config(lmax, nlat, **kw), oracle.Config(lmax, nlat, **kw)
    alm = oracle.random_alm(lmax, mmax, seed=nf, power=1.0, nf=nf)
    for m in range(mmax + 1):
        if m % mres:
            alm[:, m] = 0
    print(f"{precision} lmax={lmax} nlat={nlat} mres={mres} ltr={ltr} nf={nf}", flush=True)
    a32 = alm.astype(np.complex64)
    for dtype, a in ((torch.float64, alm), (torch.float32, a32)):
        for real in (True, False):
            got, names = _traced(cfg.plan, lambda: shtk.synthesis_batch(cfg, to_dev(a), precision=precision, ltr=ltr,
                                                                        real_output=real))
            assert names == {EVENT[precision] + "_synth", "fft_synth"}
            assert (got.real if not real else got).dtype == dtype
            ref = ocfg.synthesis(a.astype(np.complex128), ltr=ltr, real_output=real)
            assert _worst(got, ref) < (TOL[precision] if dtype == torch.float64 else 2e-6), (dtype, real)


@pytest.mark.parametrize("nlat2,graph", [(2000, False), (2050, True)])
def test_grouped_split_synthesis(shtk, oracle, cuda, nlat2, graph):
    """Two groups in split precision that both keep the split synthesis share its launches
    (no events of their own); their analyses run group by group."""
    from shtnskit_jl_amd import _lib

    shapes = [(1000, 2002, 64, 20, 16), (1023, nlat2, 48, 15, 31)]
    cfgs = [shtk.create_gauss_config(l, n, nlon=w, mmax=m) for l, n, w, m, _ in shapes]
    ocfgs = [oracle.Config(l, n, nlon=w, mmax=m) for l, n, w, m, _ in shapes]
    nfs = [s[4] for s in shapes]
    alms = [oracle.random_alm(l, m, seed=nf, power=1.0, nf=nf) for l, _, _, m, nf in shapes]
    refs = [oc.synthesis(a) for oc, a in zip(ocfgs, alms)]
    b = shtk.UnevenBatch(cfgs, nfs, precision="split", graph=graph)
    plan = ctypes.c_void_p()
    _lib.check(_lib.load().shtk_batch_plan(ctypes.c_void_p(b._b), 1, ctypes.byref(plan)), "batch_plan")
    print(f"grouped split nlat2={nlat2} graph={graph}", flush=True)
    with torch.cuda.stream(torch.cuda.Stream()):
        d = [to_dev(a) for a in alms]
        if not graph:
            fs, names = _traced(plan.value, lambda: b.synthesis(d))
            assert names == set()
        for _ in range(3):  # capture and replays
            fs = b.synthesis(d)
            backs = b.analysis(fs)
            torch.cuda.synchronize()
            for f, back, ref, a in zip(fs, backs, refs, alms):
                assert _worst(f, ref) < TOL["split"]
                assert _worst(back, a) < TOL["split"]
    b.close()


SEGMENTS = [
    # precision, lmax, nlat, nlon, mmax, mres, ltr, nf, conventions
    ("split", 3, 8, 10, None, 1, -1, 1, {}),
    ("split", 100, 128, 256, None, 1, -1, 17, {}),
    ("split", 130, 133, 264, None, 2, 101, 5, {}),
    ("split", 60, 1100, 128, None, 1, -1, 3, {}),       # two pair blocks of 512
    ("split", 40, 42, 96, None, 1, -1, 4, dict(norm="schmidt", cs_phase=False, real_norm=True)),
    ("fp32", 100, 128, 256, None, 1, -1, 17, {}),
    ("fp32", 130, 133, 264, 70, 2, 101, 5, {}),
    ("fp32", 60, 1100, 128, None, 1, -1, 3, {}),
]


@pytest.mark.parametrize("precision,lmax,nlat,nlon,mmax,mres,ltr,nf,conv", SEGMENTS)
def test_plans_of_128_degree_segments(shtk, oracle, cuda, monkeypatch, precision, lmax, nlat, nlon, mmax, mres, ltr, nf,
                                      conv):
    monkeypatch.setenv("SHTK_SEG", "128")
    mm = lmax if mmax is None else mmax
    kw = dict(nlon=nlon, mmax=mm, mres=mres, **conv)
    cfg, ocfg = shtk.create_gauss_config(lmax, nlat, **kw), oracle.Config(lmax, nlat, **kw)
    rng = np.random.default_rng(lmax + nf)
    grids = [np.asfortranarray(rng.standard_normal((nlat, nlon, nf))) for _ in range(2)]
    specs = [oracle.random_alm(lmax, mm, seed=s, power=p, nf=nf, lmin=lo) for s, p, lo in ((3, 1.0, 0), (4, 2.0, 1),
                                                                                         (5, 2.0, 1))]
    for a in specs:
        for m in range(mm + 1):
            if m % mres:
                a[:, m] = 0
    tol, ev = TOL[precision], EVENT[precision]
    print(f"segments of 128: {precision} lmax={lmax} nlat={nlat} mres={mres} ltr={ltr} nf={nf}", flush=True)
    opt = dict(precision=precision, ltr=ltr)
    got, names = _traced(cfg.plan, lambda: shtk.synthesis_batch(cfg, to_dev(specs[0]), **opt))
    assert ev + "_synth" in names and _worst(got, ocfg.synthesis(specs[0], ltr=ltr)) < tol
    got, names = _traced(cfg.plan, lambda: shtk.analysis_batch(cfg, to_dev(grids[0]), **opt))
    assert ev + "_anal" in names and _worst(got, ocfg.analysis(grids[0], ltr=ltr)) < tol
    got, names = _traced(cfg.plan, lambda: shtk.synthesis_sphtor_batch(cfg, to_dev(specs[1]), to_dev(specs[2]), **opt))
    assert "leg_synth_sphtor_low" in names  # the vector form of the matrix-core contractions
    for g, r in zip(got, ocfg.synthesis_sphtor(specs[1], specs[2], ltr=ltr)):
        assert _worst(g, r) < tol
    got = shtk.analysis_sphtor_batch(cfg, *[to_dev(g) for g in grids], **opt)
    for g, r in zip(got, ocfg.analysis_sphtor(*grids, ltr=ltr)):
        assert _worst(g, r) < tol
    a32, g32 = specs[0].astype(np.complex64), grids[0].astype(np.float32)
    assert _worst(shtk.synthesis_batch(cfg, to_dev(a32), **opt), ocfg.synthesis(a32.astype(np.complex128), ltr=ltr)) < 2e-6
    assert _worst(shtk.analysis_batch(cfg, to_dev(g32), **opt), ocfg.analysis(g32.astype(np.float64), ltr=ltr)) < 2e-6


@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_uneven_split_batch_of_128_degree_segments(shtk, oracle, cuda, monkeypatch, dtype):
    """Both directions of the grouped split kernels, one configuration with several pair blocks."""
    monkeypatch.setenv("SHTK_SEG", "128")
    shapes = [(130, 132, 264, 5), (63, 1100, 128, 17), (15, 16, 32, 1)]
    cfgs = [shtk.create_gauss_config(l, n, nlon=w) for l, n, w, _ in shapes]
    ocfgs = [oracle.Config(l, n, nlon=w) for l, n, w, _ in shapes]
    alms = [oracle.random_alm(l, l, seed=l, power=1.0, nf=nf) for l, _, _, nf in shapes]
    b = shtk.UnevenBatch(cfgs, [s[3] for s in shapes], precision="split")
    print(f"uneven split batch, segments of 128, {dtype}", flush=True)
    fs = b.synthesis([to_dev(a.astype(np.complex64 if dtype == "f32" else np.complex128)) for a in alms])
    backs = b.analysis(fs)
    tol = TOL["split"] if dtype == "f64" else 2e-6
    for f, back, oc, a in zip(fs, backs, ocfgs, alms):
        assert _worst(f, oc.synthesis(a)) < tol
        assert _worst(back, a) < 2 * tol
    b.close()
