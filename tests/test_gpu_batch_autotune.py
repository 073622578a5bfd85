"""Launch shapes an uneven batch may choose: one per direction that runs the persistent split
kernel, none (0, one timed round trip) where the FP64 field groups run."""
import numpy as np
import pytest
import torch

from _util import rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu

SMALL = [(63, 64, 128, 63, 4), (31, 32, 64, 31, 3)]
LARGE = [(1000, 2000, 32, 10, 16), (1023, 2000, 32, 8, 15)]   # both syntheses stay split


@pytest.mark.parametrize("shapes,seg,precision,synth,anal", [
    (SMALL, None, "split", False, False),
    (SMALL, None, "fp64", False, False),
    (LARGE, None, "split", True, False),
    (LARGE[:1] + SMALL[:1], None, "split", False, False),
    (SMALL, "128", "split", True, True),
])
def test_choice_follows_the_kernels(shtk, oracle, cuda, monkeypatch, shapes, seg, precision, synth, anal):
    if seg:
        monkeypatch.setenv("SHTK_SEG", seg)
    cfgs = [shtk.create_gauss_config(l, n, nlon=w, mmax=m) for l, n, w, m, _ in shapes]
    b = shtk.UnevenBatch(cfgs, [s[4] for s in shapes], precision=precision)
    alms = [oracle.random_alm(l, m, seed=l, power=1.0, nf=nf) for l, _, _, m, nf in shapes]
    print(f"autotune {shapes} seg={seg} {precision}", flush=True)
    d = [to_dev(a) for a in alms]
    choice = b.autotune([a.clone() for a in d], b.synthesis(d), reps=1)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    for key, runs in (("synth_blocks", synth), ("anal_blocks", anal)):
        assert choice[key] in ([k * cus for k in (1, 2, 3, 4)] if runs else [0]), (key, choice)
    for back, a in zip(b.analysis(b.synthesis(d)), alms):
        assert max(rel_l2(to_host(back)[..., k], a[..., k]) for k in range(a.shape[-1])) < 1e-11
    b.close()
