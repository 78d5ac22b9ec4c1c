"""The PSF blur at image sizes that leave part of a workgroup of outputs and at narrow and wide kernels, against the
oracle bit for bit."""
import numpy as np
import pytest

from gpu_util import from_dev, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,rings,psf", [(84, 17, (0.0, 0.0, 0.0)), (88, 30, (2.0, 0.0, 0.0)), (92, 16, (9.0, 30.0, 0.2)),
                                         (100, 104, (1.3, 0.0, 0.0))])
def test_convolve_and_update(oracle_lib, n, rings, psf):
    from hrrt_reconstruction_amd.osem import Osem3D
    print(f"psf runs n={n} rings={rings} psf={psf}", flush=True)
    geom = dict(rings=rings, def_elements=n, def_angles=48, x_pixels=n, span=3, maxdel=5, z_min=3, z_max=2 * rings - 4,
                subsets=4)
    o, g = oracle_lib.Oracle(**geom), Osem3D(**geom)
    o.set_psf(*psf)
    g.set_psf(*psf)
    rng = np.random.default_rng(n)
    img = np.ascontiguousarray(o.init_image() * rng.uniform(0.0, 2.0, (o.N, o.N, o.Z4)).astype(np.float32))
    assert np.array_equal(from_dev(g.convolve3d(to_dev(img))), o.convolve3d(img))
    shape = (o.S, o.views, o.N)
    prompt = rng.integers(0, 4, shape).astype(np.int16)
    add = rng.uniform(0.0, 0.2, shape).astype(np.float32)
    nf = rng.uniform(0.05, 2.0, (o.subsets, o.N, o.N, o.Z4)).astype(np.float32)
    d_img = to_dev(img)
    g.osem_subset(d_img, to_dev(nf), to_dev(g.sino_to_paircol(prompt)), to_dev(g.sino_to_paircol(add)), 1)
    o.osem_subset_psf(img, o.image_zeros(), np.ascontiguousarray(nf[1]), add, prompt, 1, nthreads=g.backproject_schedule,
                      workers=4)
    assert np.array_equal(from_dev(d_img), img)
