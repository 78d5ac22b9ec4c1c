"""A batch of frames in the precision form against its single frames: images and log-likelihoods bit for bit,
and the log-likelihood's sum over terms of every size.

The geometries have fewer than 512 rays (view pairs x half the bins) in a frame and more in the batch, the
line at which the forward projector's launch shape changes: span 9 at 128 x 128 goes from one plane to a
run of three per thread and from 16 waves to fewer, the 16-ring scanner from 16 waves to 4.  The
header promises the frame's values for the batch, and a log-likelihood that does not depend on the shape.
"""
import math

import numpy as np
import pytest

import bruteforce as bf
from conftest import GEOMS
from gpu_util import from_dev, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("geom,frames", [("tiny9", 4), ("c1", 8)])
@pytest.mark.parametrize("loglik", [False, True])
def test_batch_equals_frames(geom, frames, loglik):
    import torch
    from hrrt_reconstruction_amd.osem import Osem3D
    print(f"frames loglik geom={geom} frames={frames} loglik={loglik}", flush=True)
    g = Osem3D(**GEOMS[geom])
    rays = g.N // 2 * (g.views // g.subsets // 2)
    assert rays < 512 <= rays * frames
    gen = torch.Generator(device="cuda")
    gen.manual_seed(90)

    def uniform(shape, lo, hi):
        return torch.rand(shape, generator=gen, device="cuda") * (hi - lo) + lo

    cols = (g.views // 2, 2, g.N, g.spp)
    pr = torch.poisson(uniform((frames,) + cols, 0.0, 3.0), generator=gen).to(torch.int16)
    add = g.to_half(uniform((frames,) + cols, 0.01, 0.3))
    inv = g.to_half(uniform(cols, 0.5, 1.5))
    nf = uniform((g.subsets, g.N, g.N, g.Z4), 0.05, 2.0)
    batch = torch.stack([g.init_image() * (1 + f) for f in range(frames)])
    single = batch.clone()
    llb = torch.zeros(frames, dtype=torch.float64, device="cuda")
    lls = torch.zeros(frames, dtype=torch.float64, device="cuda")
    # two orders of one double sum mostly round to the same total: every subset, so that one of them tells
    for s in range(g.subsets if loglik else 2):
        g.osem_subset_frames_mixed(batch, nf, pr, add, s, invnorm16=inv, loglik=llb if loglik else None)
        for f in range(frames):
            g.osem_subset_mixed(single[f], nf, pr[f], add[f], s, invnorm16=inv, loglik=lls[f:f + 1] if loglik else None)
        assert np.array_equal(from_dev(batch), from_dev(single)), s
        assert np.array_equal(from_dev(llb), from_dev(lls)), (s, llb.tolist(), lls.tolist())
        assert not loglik or np.all(np.isfinite(from_dev(llb))) and np.all(from_dev(llb) != 0)
        if loglik and s == 0:
            for shape in ((1, 3), (3, 1), (3, 2)):
                g.set_launch_shape(*shape)
                lls.zero_()
                again = g.init_image()[None] * torch.arange(1.0, frames + 1, device="cuda")[:, None, None, None]
                g.osem_subset_frames_mixed(again, nf, pr, add, s, invnorm16=inv, loglik=lls)
                assert np.array_equal(from_dev(llb), from_dev(lls)), shape
            g = Osem3D(**GEOMS[geom])


@pytest.mark.parametrize("scale", [1.0, 1e8])
def test_sum_of_terms(oracle_lib, scale):
    """Against the exact sum of the float64 terms.  A term carries the rounding of its logarithm and of itself, a few
    2^-53 of it, so 1e-14 of the sum of magnitudes; at the larger scale some means lie above 2^32 and some below."""
    import torch
    from hrrt_reconstruction_amd.osem import Osem3D
    print(f"loglik terms scale={scale}", flush=True)
    o, g, G = oracle_lib.Oracle(**GEOMS["tiny"]), Osem3D(**GEOMS["tiny"]), bf.Geometry(**GEOMS["tiny"])
    rng = np.random.default_rng(91)
    shape = (o.S, o.views, o.N)
    inv = (0.5 * 10.0 ** rng.uniform(0.0, 2.0, shape)).astype(np.float16).astype(np.float32)
    add = rng.uniform(0.1, 0.5, shape).astype(np.float16).astype(np.float32)
    prompt = rng.poisson(2.0, shape).astype(np.int16)
    img = (scale * rng.uniform(0.5, 1.5, (o.N, o.N, o.Z4))).astype(np.float32)
    s = 5
    d_img, d_pr = to_dev(img), to_dev(g.sino_to_paircol(prompt))
    d_add, d_inv = g.to_half(to_dev(g.sino_to_paircol(add))), g.to_half(to_dev(g.sino_to_paircol(inv)))
    nf = torch.ones((o.subsets, o.N, o.N, o.Z4), device="cuda")
    ll = torch.zeros(1, dtype=torch.float64, device="cuda")
    terms = []
    fov = np.array([x > 0 and G.cyl[x][0] != G.cyl[x][1] for x in range(o.N)])
    for v in o.vieworder[s][: o.sviews // 2]:
        den = from_dev(g.forward_proj3d(d_img, v)) + bf.gather_pair(add, v)
        w, y = (bf.gather_pair(t, v).astype(np.float64) for t in (inv, prompt))
        ok = (w > 0) & (den > o.params.epsilon3) & fov[None, :]
        mu = np.where(ok, den.astype(np.float64) * w, 1.0)
        terms.append((np.where(y > 0, y * np.log(mu), 0.0) - mu)[ok])
    terms = np.concatenate(terms)
    assert (np.abs(terms) < 2.0 ** 32).any() and (scale == 1.0 or (np.abs(terms) > 2.0 ** 32).any())
    g.osem_subset_mixed(d_img.clone(), nf, d_pr, d_add, s, invnorm16=d_inv, loglik=ll)
    exact, size = math.fsum(terms), math.fsum(np.abs(terms))
    got = float(ll.item())
    print(f"loglik {got:.17g} exact {exact:.17g} error {(got - exact) / size:.2e} of the magnitudes", flush=True)
    assert abs(got - exact) <= 1e-14 * size
    # a bin without prompts whose mean is infinite, in a view of the subset
    add[o.S // 2, o.vieworder[s][0], o.N // 2 + 3] = np.inf
    prompt[o.S // 2, o.vieworder[s][0], o.N // 2 + 3] = 0
    g.osem_subset_mixed(d_img.clone(), nf, to_dev(g.sino_to_paircol(prompt)), g.to_half(to_dev(g.sino_to_paircol(add))), s,
                        invnorm16=d_inv, loglik=ll)
    assert ll.item() == -math.inf
