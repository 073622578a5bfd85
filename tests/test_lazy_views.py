"""Arrays handed to the library hold the tensor's values: torch's lazy conjugate and negative
views (also the cotangents of a conjugation) share memory with the values before."""
import pytest
import torch

from _util import rel_l2, to_dev, to_host


def test_memory_holds_the_values(shtk):
    from shtnskit_jl_amd.transforms import _colmajor

    z = torch.randn(4, 3, 2, dtype=torch.complex128)
    base = z.permute(2, 1, 0).contiguous().permute(2, 1, 0)  # column-major already
    for t in (base.conj(), z.conj(), base.conj().imag, z.conj().imag):
        c = _colmajor(t)
        assert not c.is_conj() and not c.is_neg()
        assert torch.equal(c, t.resolve_conj().resolve_neg())
        assert c.stride() == (1, 4, 12)
    assert _colmajor(base) is base


@pytest.mark.gpu
def test_conjugate_views_on_the_device(shtk, oracle, cuda):
    lmax, nlat, nlon = 20, 22, 42
    cfg, ocfg = shtk.create_gauss_config(lmax, nlat, nlon=nlon), oracle.Config(lmax, nlat, nlon=nlon)
    alm = oracle.random_alm(lmax, lmax, seed=1, power=1.0)
    got = shtk.synthesis(cfg, to_dev(alm).conj())
    assert rel_l2(to_host(got), ocfg.synthesis(alm.conj())) < 1e-12
    # a loss whose cotangent is a conjugate view
    f = to_dev(ocfg.synthesis(alm)).requires_grad_()
    z = to_dev(oracle.random_alm(lmax, lmax, seed=2, power=1.0))
    (shtk.ad.analysis(cfg, f).conj() * z).real.sum().backward()
    assert rel_l2(to_host(f.grad), ocfg.adjoint_analysis(to_host(z)).real) < 1e-12
