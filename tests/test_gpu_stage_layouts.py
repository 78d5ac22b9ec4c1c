"""Staging: 16-byte loads and stores against the element-wise form, on files and outputs at odd addresses."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


# radial bins that end inside a tile, rebinned or not, end planes of every kind
@pytest.mark.parametrize("weighting", [3, 0, 1, 2])
@pytest.mark.parametrize("rings,bins,angles,x", [(9, 84, 96, 84), (9, 176, 176, 88), (21, 240, 240, 80)])
def test_stage_layouts(weighting, rings, bins, angles, x):
    import torch
    from hrrt_reconstruction_amd import _lib
    from hrrt_reconstruction_amd.osem import Osem3D
    print(weighting, rings, bins, angles, x, flush=True)
    g = Osem3D("cuda:0", rings=rings, def_elements=bins, def_angles=angles, x_pixels=x, span=3, maxdel=4, subsets=8,
               z_min=3, z_max=2 * rings - 4)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(rings)
    shape = (g.S, angles, bins)
    u = lambda lo, hi: torch.rand(shape, generator=gen, device="cuda") * (hi - lo) + lo  # noqa: E731
    norm = u(0.5, 1.5) * (torch.rand(shape[1:], generator=gen, device="cuda") > 0.1)
    norm[:, :, 5] = 0
    prompt = torch.randint(0, 9, shape, generator=gen, device="cuda", dtype=torch.int16)
    files = [prompt, u(0, 1), norm, u(0, 2), u(0.5, 3)]

    def moved(t):                # the same values one element further on
        o = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")[1:].view(t.shape)
        o.copy_(t)
        return o

    def stage(f):
        outs = g.stage(*f) if weighting == 3 else g.stage_w012(weighting, *f)
        return list(outs), g.norm_zero_mask()

    ref, mask = stage(files)
    pads = torch.ones(g.spp, dtype=torch.bool, device="cuda")
    for s in range(g.th):
        pads[int(g.seg_data[s]):int(g.seg_data[s] + g.yr_top[s] - g.yr_bottom[s] + 1)] = False
    for t in ref:
        assert int(torch.count_nonzero(t[..., pads])) == 0      # guard planes
    got, m = stage([moved(t) for t in files])
    assert (m == mask).all()
    for a, b in zip(got, ref):
        assert torch.equal(a, b)
    # outputs at odd addresses, full of other values before
    outs = [moved(torch.full_like(t, 7)) for t in ref]
    ptr = [C.c_void_p(t.data_ptr()) for t in files]
    out = [C.c_void_p(t.data_ptr()) for t in outs]
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    if weighting == 3:
        _lib.call("hrrt_stage_sinograms", g.ctx, *ptr, *out, stream)
    else:
        _lib.call("hrrt_stage_sinograms_w012", g.ctx, weighting, 0, ptr[0], C.c_void_p(0), *ptr[1:], *out, stream)
    for a, b in zip(outs, ref):
        assert torch.equal(a, b)
