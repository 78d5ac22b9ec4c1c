"""Launch-shape autotuner for the projectors.

The forward projector's workgroup owns planes of one ray column (one x of
one view pair); the shape picks whether each thread accumulates one plane or a
run of three, and how many workgroups share one column (each recomputing the
column's rotated samples).  The back
projector's workgroup stages one sinogram column in LDS; its shape is the
number of waves (voxel rows in flight) sharing that column.  Results are
bit-identical for every shape; only speed differs.  The choice between the
incremental and the direct back projector is not a shape: the two differ by
float rounding, as they do in the reference, and that choice stays with the
caller (hrrt_set_backproject_schedule, the reference's -T).  The tuner times the
candidates on the caller's own subset update with HIP events and keeps the
fastest; tune_frames does the same on the batched update of every frame of a
dynamic study, whose forward launches have a frame dimension of their own.
"""
from __future__ import annotations

# (0, 0) leaves both numbers to each launch's count of rays and planes; the others fix them for every call
CANDIDATES = [(0, 0), (1, 0), (1, 3), (1, 4), (1, 6), (3, 0), (3, 2), (3, 3)]
BY_RULE_MARGIN = 0.05


def _choose(results):
    """The fastest shape, but (0, 0) unless another is faster by more than repeated timings differ: a fixed shape
    also holds for the context's calls of other sizes, where it may be the slower one."""
    best = min(results, key=results.get)
    rule = (0, 0)
    return rule if rule in results and results[rule] <= (1 + BY_RULE_MARGIN) * results[best] else best


BP_CANDIDATES = [4, 8, 12, 16]


def _time_kernel(g, work, normfac, prompt, add, subsets, repeats, kernel):
    import torch
    g.osem_subset(work, normfac, prompt, add, subsets[0])      # warm-up / first launch of this variant
    torch.cuda.synchronize()
    g.timing_enable(True)
    for _ in range(repeats):
        for s in subsets:
            g.osem_subset(work, normfac, prompt, add, s)
    kt = g.timing_read()
    g.timing_enable(False)
    ms, n = kt[kernel]
    return ms / max(n, 1)


def tune_backproject(g, image, normfac, prompt, add, subsets=(0, 8), repeats=2, candidates=BP_CANDIDATES):
    """Choose the direct back projector's workgroup size (waves per workgroup).

    Workgroup sizes give bit-identical results; only speed differs.  The direct projector
    serves the remainder pairs of a -T schedule, schedule 0 and the precision form, so it
    is timed under schedule 0.  The caller's back-projection schedule (the reference's
    -T, which decides per pair between the incremental and the direct projector and with
    it the float rounding) is restored before returning, and its own back-projection
    time is reported as "schedule T=<n>".  The tuner never changes the algorithm.
    Returns (waves, {label: ms per back-projection launch})."""
    work = image.clone()
    results = {}
    keep = g.backproject_schedule
    try:
        g.set_backproject_schedule(0)
        for w in candidates:
            g.set_backproject_shape(w)
            results[f"direct/{w}w"] = _time_kernel(g, work, normfac, prompt, add, subsets, repeats, "backproject")
        best_w = min(candidates, key=lambda w: results[f"direct/{w}w"])
        g.set_backproject_shape(best_w)
    finally:
        g.set_backproject_schedule(keep)
    if keep != 0:
        results[f"schedule T={keep}"] = _time_kernel(g, work, normfac, prompt, add, subsets, repeats, "backproject")
    del work
    return best_w, results


def _forward_times(g, step, subsets, repeats, candidates):
    """{shape: ms per forward launch}, the least of `repeats` rounds over all candidates (the first ones meet a GPU whose
    clock still rises: one after the other, two shapes of the same kernel came out 10 % apart)."""
    import torch
    results = {}
    for _ in range(repeats):
        for shape in candidates:
            try:
                g.set_launch_shape(*shape)
            except Exception:
                continue
            step(subsets[0])                      # warm-up / first launch of this variant
            torch.cuda.synchronize()
            g.timing_enable(True)
            for s in subsets:
                step(s)
            ms, n = g.timing_read()["fp_ratio"]
            g.timing_enable(False)
            results[shape] = min(results.get(shape, float("inf")), ms / max(n, 1))
    return results


def tune_forward(g, image, normfac, prompt, add, subsets=(0, 8), repeats=2, candidates=CANDIDATES):
    """Return ((tasks_per_thread, workgroups_per_ray), {shape: ms per forward launch})."""
    work = image.clone()
    results = _forward_times(g, lambda s: g.osem_subset(work, normfac, prompt, add, s), subsets, repeats, candidates)
    best = _choose(results)
    g.set_launch_shape(*best)
    return best, results


def tune_frames(g, images, normfac, prompts, adds, mixed=False, subsets=(0, 8), repeats=2, candidates=CANDIDATES):
    """Forward launch shape for the batched path (hrrt_osem_subset_frames, or the FP16-input
    form with mixed=True): every candidate timed on subset updates of all frames, the
    fastest kept on the context.  Shapes give bit-identical results; a new shape drops the
    context's captured iteration graphs, which the next iteration call captures again.
    Returns ((tasks_per_thread, workgroups_per_ray), {shape: ms per forward launch})."""
    work = images.clone()
    update = g.osem_subset_frames_mixed if mixed else g.osem_subset_frames
    results = _forward_times(g, lambda s: update(work, normfac, prompts, adds, s), subsets, repeats, candidates)
    best = _choose(results)
    g.set_launch_shape(*best)
    return best, results
