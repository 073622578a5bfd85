"""An infinity or NaN in one field of a batch: the field groups spoil exactly the coefficients
that the single-field kernel spoils (those whose Legendre values are live at that row) and no
other field's."""
import numpy as np
import pytest
import torch

from _util import rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lmax,nlat,row", [(200, 202, 0), (200, 202, 3), (200, 202, 201), (511, 512, 0), (511, 512, 256)])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_rows_that_count_for_nothing(shtk, cuda, monkeypatch, lmax, nlat, row, value):
    # the longitude transform packs two rows of a tile into one: the same tiles for both calls
    monkeypatch.setenv("SHTK_FFT_PAIRS", "4")
    nlon, nf, bad = 2 * lmax + 2, 8, 3
    cfg = shtk.create_gauss_config(lmax, nlat, nlon=nlon)
    f = np.random.default_rng(lmax).standard_normal((nlat, nlon, nf))
    f[row, 1, bad] = value
    print(f"lmax={lmax} row={row} {value}", flush=True)
    for call in (shtk.analysis_batch, shtk._adjoint_synthesis):
        got = to_host(call(cfg, to_dev(f)))
        one = to_host(call(cfg, to_dev(f[..., bad:bad + 1])))[..., 0]
        assert not np.isfinite(one).all()
        assert np.array_equal(np.isfinite(got[..., bad]), np.isfinite(one))
        live = np.isfinite(one)
        assert rel_l2(got[..., bad][live], one[live]) < 1e-12
        rest = [k for k in range(nf) if k != bad]
        assert np.isfinite(got[..., rest]).all()
