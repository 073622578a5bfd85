"""Work items of the single-field analysis kernel, whose list holds the segments of the
degrees to lmax first and those of the degree lmax + 1 alone (vector transforms) behind
them: lmax + 1 a multiple of 64, where the last segment of some orders is such a one, one
and several pair blocks, with the outputs handed over full of NaN.  FP64, so the bound is
the FP64 path's 1e-12 relative L2."""
import ctypes

import numpy as np
import pytest

from _util import rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu

TOL = 1e-12

SHAPES = [
    # lmax, nlat, nlon, mres, ltr, nf
    (62, 64, 126, 1, -1, 1),
    (63, 64, 128, 1, -1, 1),
    (63, 1100, 128, 1, -1, 2),     # two pair blocks, sums added in memory
    (64, 66, 130, 1, 63, 3),
    (127, 129, 256, 2, -1, 1),
    (191, 192, 384, 3, 128, 2),
    (255, 256, 512, 1, -1, 3),
]


def _nan_outputs(cfg, nf, n):
    import torch

    return [torch.full((nf, cfg.mmax + 1, cfg.lmax + 1), complex(float("nan"), float("nan")), dtype=torch.complex128,
                       device="cuda:0").permute(2, 1, 0) for _ in range(n)]


@pytest.mark.parametrize("lmax,nlat,nlon,mres,ltr,nf", SHAPES)
def test_analyses_match_oracle(shtk, oracle, cuda, lmax, nlat, nlon, mres, ltr, nf):
    from shtnskit_jl_amd import _lib
    from shtnskit_jl_amd.transforms import _ptr, _stream

    cfg = shtk.create_gauss_config(lmax, nlat, nlon=nlon, mres=mres)
    ocfg = oracle.Config(lmax, nlat, nlon=nlon, mres=mres)
    rng = np.random.default_rng(lmax + nlat)
    f, g = [np.asfortranarray(rng.standard_normal((nlat, nlon, nf))) for _ in range(2)]
    fd, gd = to_dev(f), to_dev(g)
    plan, lib, st = ctypes.c_void_p(cfg.plan), _lib.load(), _stream(fd.device)
    print(f"lmax={lmax} nlat={nlat} mres={mres} ltr={ltr} nf={nf}", flush=True)
    (out,) = _nan_outputs(cfg, nf, 1)
    _lib.check(lib.shtk_analysis(plan, _ptr(fd), _ptr(out), nf, _lib.SHTK_F64, ltr, st), "analysis")
    vec = _nan_outputs(cfg, nf, 2)
    _lib.check(lib.shtk_analysis_sphtor(plan, _ptr(fd), _ptr(gd), _ptr(vec[0]), _ptr(vec[1]), nf, _lib.SHTK_F64, ltr,
                                        st), "analysis_sphtor")
    refs = [ocfg.analysis(f, ltr=ltr), *ocfg.analysis_sphtor(f, g, ltr=ltr)]
    for got, ref in zip([out, *vec], refs):
        got = to_host(got)
        assert max(rel_l2(got[..., k], ref[..., k]) for k in range(nf)) < TOL
        assert np.all(got[ref == 0] == 0)
