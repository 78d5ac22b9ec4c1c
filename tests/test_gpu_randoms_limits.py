"""Smoothed randoms at the limits of float."""
import pytest

pytestmark = pytest.mark.gpu


def test_overflowing_factor_of_silent_crystals():
    """singles * tau * T overflows for one crystal column and every other crystal is silent: all terms are zero."""
    import torch
    from hrrt_reconstruction_amd.randoms import GenDelays
    print("randoms overflowing factor", flush=True)
    s = torch.zeros((2, 104, 8, 72), device="cuda")     # [layer][ring][head][x]
    s[1, :, 0, 30] = 1e38
    g = GenDelays(span=9, lr_type=2)
    out = g.smooth(s.reshape(-1), 1e10)                 # tau * T = 60
    assert not out.any().item()
