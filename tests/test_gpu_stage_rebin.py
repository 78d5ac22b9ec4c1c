"""Staging against the oracle, files at any element's address: rows read in groups of four (no rebinning, 2 x 2) and
bin by bin (3 x 3)."""
import numpy as np
import pytest

from gpu_util import from_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bins,angles,x", [(84, 96, 84), (176, 176, 88), (240, 240, 80)])
@pytest.mark.parametrize("shift", [0, 1, 2])
def test_stage_rebin(oracle_lib, bins, angles, x, shift):
    import torch
    from hrrt_reconstruction_amd.osem import Osem3D
    print(f"stage rebin {bins}x{angles} -> {x}, {shift} elements off", flush=True)
    geom = dict(rings=9, def_elements=bins, def_angles=angles, x_pixels=x, span=3, maxdel=4, subsets=8, z_min=3, z_max=14)
    o, g = oracle_lib.Oracle(**geom), Osem3D("cuda:0", **geom)
    shape = (o.S, angles, bins)
    rng = np.random.default_rng(bins)
    u = lambda lo, hi: rng.uniform(lo, hi, shape).astype(np.float32)  # noqa: E731
    norm = u(0.5, 1.5)
    norm[:, rng.random(shape[1:]) < 0.1] = 0
    norm[:, :, 5] = 0
    files = [rng.integers(0, 9, shape).astype(np.int16), u(0, 1), norm, u(0, 2), u(0.5, 3)]

    def moved(a):
        t = torch.from_numpy(a)
        d = torch.empty(t.numel() + shift, dtype=t.dtype, device="cuda")[shift:].view(t.shape)
        d.copy_(t)
        return d

    dev = [moved(a) for a in files]
    ref_inv = o.prepare_norm(files[2], files[4])
    ref_pr, ref_add = o.prepare_w3(*files)
    pr, add, inv = g.stage(*dev)
    for got, ref in ((pr, ref_pr), (add, ref_add), (inv, ref_inv)):
        assert np.array_equal(from_dev(got), g.sino_to_paircol(ref))
    ref_data = o.prepare_w012(1, files[0], files[1], files[2], files[3], files[4])
    data, inv = g.stage_w012(1, *dev)
    assert np.array_equal(from_dev(data), g.sino_to_paircol(ref_data))
    assert np.array_equal(from_dev(inv), g.sino_to_paircol(o.prepare_norm_w(1, files[2], files[4])))
