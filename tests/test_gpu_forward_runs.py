"""Forward projector: runs of planes, singles and launch shapes at their edges, against the oracle."""
import numpy as np
import pytest

from gpu_util import from_dev, to_dev
from oracle import oracle

pytestmark = pytest.mark.gpu

# (rings, radial bins, span, maxdel): group sizes of every remainder modulo 3, groups shorter than a run,
# one to four sample chunk groups per half row, planes below and above 4, 8 and 16 waves
GEOMS = [(8, 80, 3, 4), (11, 80, 3, 7), (16, 84, 9, 13), (33, 80, 3, 16), (70, 80, 9, 40), (104, 80, 3, 31), (128, 80, 3, 60)]


@pytest.mark.parametrize("rings,bins,span,maxdel", GEOMS)
def test_forward_runs(oracle_lib, rings, bins, span, maxdel):
    import torch
    from hrrt_reconstruction_amd.osem import Osem3D
    geom = dict(rings=rings, def_elements=bins, def_angles=48, x_pixels=bins, span=span, maxdel=maxdel, subsets=8,
                z_min=3, z_max=2 * rings - 4)
    print(geom, flush=True)
    o = oracle.Oracle(**geom)
    g = Osem3D("cuda:0", **geom)
    rng = np.random.default_rng(rings)
    img = np.ascontiguousarray(o.init_image() * rng.uniform(0.5, 2.0, (o.N, o.N, o.Z4)).astype(np.float32))
    ref = o.forward(img, 5)
    for shape in (None, (1, 0), (3, 0), (4, 3)):
        if shape:
            g.set_launch_shape(*shape)
        assert np.array_equal(from_dev(g.forward_proj3d(to_dev(img), 5)), ref), shape
    # one subset of enough frames for workgroups of as few waves as the planes need: each equals the
    # frame alone
    g = Osem3D("cuda:0", **geom)
    frames = 512 // (o.N // 2 * (o.views // 16)) + 1
    d_img = torch.stack([to_dev(img) * (1 + f) for f in range(frames)])
    pr = torch.randint(0, 4, (frames, g.views // 2, 2, g.N, g.spp), device="cuda", dtype=torch.int16)
    add = torch.rand(pr.shape, device="cuda") + 0.01
    nf = torch.rand((g.subsets, g.N, g.N, g.Z4), device="cuda")
    one = d_img.clone()
    g.osem_subset_frames(d_img, nf, pr, add, 3)
    for f in range(frames):
        g.osem_subset(one[f], nf, pr[f], add[f], 3)
    assert np.array_equal(from_dev(d_img), from_dev(one))
