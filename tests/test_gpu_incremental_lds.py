"""Incremental back projector whose columns of two bins take more than 64 KB of LDS, against the oracle."""
import numpy as np
import pytest

from gpu_util import from_dev, to_dev
from oracle import oracle
from test_gpu_incremental_layouts import GEOMS as LAYOUTS

pytestmark = pytest.mark.gpu


def _geometry(rings, bins, span, maxdel, subsets):
    return dict(rings=rings, def_elements=bins, def_angles=48, x_pixels=bins, span=span, maxdel=maxdel,
                subsets=subsets, z_min=3, z_max=2 * rings - 4)


# 128 rings at span 3: both bins of a ray take 69.6 KB of cells at 67 ring differences, two workgroups per CU, and
# 83.2 KB at 97, where twelve view pairs get a bin per workgroup as three do
@pytest.mark.parametrize("maxdel", [67, 97])
@pytest.mark.parametrize("subsets", [8, 2])
def test_large_columns(oracle_lib, maxdel, subsets):
    from hrrt_reconstruction_amd.osem import Osem3D
    geom = _geometry(128, 80, 3, maxdel, subsets)
    print(geom, flush=True)
    o, g = oracle.Oracle(**geom), Osem3D("cuda:0", **geom)
    assert g.backproject_schedule == 1
    inv = np.random.default_rng(maxdel).uniform(0.5, 1.5, (o.S, o.views, o.N)).astype(np.float32)
    ref = o.calculate_normfac(inv.copy(), nthreads=1)
    got = from_dev(g.calculate_normfac(to_dev(g.sino_to_paircol(inv))))
    assert np.array_equal(got, np.asarray(ref).reshape(got.shape))


@pytest.mark.parametrize("geom", LAYOUTS)
def test_layout_geometries_are_incremental(geom):
    from hrrt_reconstruction_amd.osem import Osem3D
    print(geom, flush=True)
    assert Osem3D("cuda:0", **_geometry(*geom)).backproject_schedule == 1
