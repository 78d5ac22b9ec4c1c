"""List mode with runs of out-of-sync words (zeros), which the walk takes 64 at a time, against the oracle."""
import numpy as np
import pytest

from hrrt_reconstruction_amd.phantom import lm_synthetic_stream
from oracle import oracle as O
from test_gpu_lmhist import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lengths", [(63, 64, 65, 127, 128, 129), (191, 2047, 2048, 2049, 1, 4097), (100_001, 62, 1984)])
@pytest.mark.parametrize("front", [0, 1, 2])
def test_zero_runs(lengths, front):
    import torch
    from hrrt_reconstruction_amd.randoms import GenDelays
    print(f"lmhist zero runs {lengths} behind {front}", flush=True)
    w = lm_synthetic_stream(20_000, 17, events_per_ms=500)
    rng = np.random.default_rng(sum(lengths) + front)
    cuts = np.sort(rng.integers(0, w.size // 2, len(lengths))) * 2
    cuts[0] = 0
    parts = [np.zeros(front, np.uint32)]
    for a, b, n in zip(cuts, list(cuts[1:]) + [w.size], lengths):
        parts += [w[a:b], np.zeros(n, np.uint32)]
    words = np.concatenate(parts)
    st = _check(torch, GenDelays(span=9), O.Delays(span=9), words, torch.from_numpy(words.view(np.int32)).cuda(), mode=1)
    assert st["events"] > 15_000


def test_nothing_but_zeros():
    import torch
    from hrrt_reconstruction_amd.randoms import GenDelays
    print("lmhist zeros", flush=True)
    words = np.zeros(2 ** 21 + 4095, np.uint32)
    st = _check(torch, GenDelays(span=9), O.Delays(span=9), words, torch.from_numpy(words.view(np.int32)).cuda())
    assert st["events"] == 0
