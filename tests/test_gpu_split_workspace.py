"""Device memory of split syntheses: the workspace of the direction that runs, not of the
analysis, which 64-degree plans never contract in split precision."""
import numpy as np
import pytest
import torch

from _util import rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu


def _first_split_call(shtk, nf, dtype):
    """Bytes a plan's first split synthesis takes beyond the FP64 workspace."""
    lmax, nlat, nlon, mmax = 1000, 2000, 202, 100
    cfg = shtk.create_gauss_config(lmax, nlat, nlon=nlon, mmax=mmax)
    rng = np.random.default_rng(3)
    a = rng.standard_normal((lmax + 1, mmax + 1, nf)) + 1j * rng.standard_normal((lmax + 1, mmax + 1, nf))
    a *= (np.arange(lmax + 1)[:, None] >= np.arange(mmax + 1))[..., None]
    a[:, 0] = a[:, 0].real
    d = to_dev(a.astype(dtype))
    ref = shtk.synthesis_batch(cfg, d)
    out = torch.empty_like(ref)
    del out
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    got = shtk.synthesis_batch(cfg, d, precision="split")  # its output reuses the freed block
    torch.cuda.synchronize()
    grown = before - torch.cuda.mem_get_info()[0]
    assert rel_l2(to_host(got[..., 0]), to_host(ref[..., 0])) < (1e-11 if dtype == np.complex128 else 1e-6)
    cfg.close()
    return grown


def test_split_synthesis_workspace(shtk, cuda):
    nf = 48
    print("split synthesis workspace", flush=True)
    _first_split_call(shtk, 16, np.complex128)  # loads the kernels
    grown = [_first_split_call(shtk, nf, dtype) for dtype in (np.complex128, np.complex64)]
    print([g >> 20 for g in grown], "MiB", flush=True)
    acc = nf * 1001 * 101 * 16  # FP64 coefficients, which only an analysis accumulates
    assert abs(grown[1] - grown[0]) < acc // 2
