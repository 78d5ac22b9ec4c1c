"""Smoothed randoms at the edges of the ring window and of the LOR batches, against the oracle.

Windows of 30 and 31 rings skip the middle ring differences and 32 does not; LR type 2 has bins
of more LORs than one batch holds.  The sums are exact in fixed point and the oracle adds in
float, so the tolerance is that of the smoothing tests: 2e-5 per element covers n 2^-24 for the
n <= 300 terms of an element.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

RTOL = 2e-5


@pytest.mark.parametrize("span,lr_type,maxrd", [(3, 0, 25), (3, 2, 26), (3, 2, 27), (9, 1, 45)])
def test_window_edges(span, lr_type, maxrd):
    import torch
    from hrrt_reconstruction_amd.randoms import GenDelays
    print(f"randoms window span={span} lr={lr_type} maxrd={maxrd}", flush=True)
    rng = np.random.default_rng(maxrd)
    s = rng.uniform(20.0, 200.0, O.NCRYS).astype(np.float32)
    s[rng.random(O.NCRYS) >= 0.05] = 0.0
    out = GenDelays(span=span, maxrd=maxrd, lr_type=lr_type).smooth(torch.from_numpy(s).cuda(), 600.0).cpu().numpy()
    ref, pairs = O.Delays(span=span, maxrd=maxrd, lr_type=lr_type).smooth(s, 6e-9, 600.0)
    assert pairs > 0 and out.shape == ref.shape
    assert np.array_equal(out == 0, ref == 0)
    assert np.all(np.abs(out - ref) <= RTOL * np.abs(ref))


def test_nan_singles_contribute_nothing():
    import torch
    from hrrt_reconstruction_amd.randoms import GenDelays
    print("randoms NaN singles", flush=True)
    rng = np.random.default_rng(3)
    s = torch.from_numpy(rng.uniform(20.0, 200.0, O.NCRYS).astype(np.float32)).cuda()
    dead = torch.from_numpy(rng.random(O.NCRYS) < 0.01).cuda()
    g = GenDelays(span=9, lr_type=2)
    a = g.smooth(s.masked_fill(dead, float("nan")), 60.0)
    assert torch.equal(a, g.smooth(s.masked_fill(dead, 0.0), 60.0))
