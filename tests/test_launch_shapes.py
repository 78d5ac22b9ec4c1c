"""The forward projector's launch shapes: the tuner's list and choice, and the way back to the library's rule."""
import numpy as np
import pytest

from conftest import GEOMS


def test_candidates_launch_different_kernels():
    from hrrt_reconstruction_amd.autotune import CANDIDATES
    launched = [(0 if tasks == 0 else 1 if tasks < 3 else 3, split) for tasks, split in CANDIDATES]
    assert len(set(launched)) == len(CANDIDATES) and CANDIDATES[0] == (0, 0)


@pytest.mark.parametrize("times,choice", [
    ({(0, 0): 1.0, (3, 0): 0.995, (1, 0): 1.3}, (0, 0)),
    ({(0, 0): 1.0, (3, 0): 0.9, (1, 0): 1.3}, (3, 0)),
    ({(3, 0): 1.0, (1, 0): 0.999}, (1, 0)),
])
def test_choice(times, choice):
    from hrrt_reconstruction_amd.autotune import _choose
    assert _choose(times) == choice


@pytest.mark.gpu
def test_back_to_the_rule():
    import torch
    from hrrt_reconstruction_amd import _lib
    from hrrt_reconstruction_amd.osem import Osem3D
    print("launch shape back to the rule", flush=True)
    g = Osem3D(**GEOMS["tiny"])
    img = g.init_image()
    ref = g.forward_proj3d(img, 7).cpu().numpy()
    for shape in ((3, 2), (0, 3), (0, 0)):
        g.set_launch_shape(*shape)
        assert np.array_equal(g.forward_proj3d(img, 7).cpu().numpy(), ref), shape
    for shape in ((-1, 0), (5, 0), (0, -1), (0, 65)):
        with pytest.raises(_lib.HrrtError, match="out of range"):
            g.set_launch_shape(*shape)
    torch.cuda.synchronize()
