"""The masked methods' passes from kept step bits, where the bits can go
wrong: segments of up to 46 steps (three words of 16) and of one voxel, runs
that break and restart at every few steps (half the voxels masked, or a
threshold at the median curl), both readings of Select's per-axis rule, edges
of tiles in every axis.  Against the walk with one lane per ray, which asks
the rule at every step: visit counts exact; p and curl weights are the same
terms in another order (FP64 1e-12, curl quotients 1e-10; FP32 ray sums 1e-5).
"""
import numpy as np
import pytest

import omni3d
import oracle as O
from omni3d import fields as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(17, 33, 16), (2, 5, 40)])
# (the per-axis rule that `faithful` asks for is Select's)
@pytest.mark.parametrize("method,faithful", [("plain", 0), ("mask", 0), ("select", 0),
                                             ("select", 1), ("weighted", 0)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("solver", ["affine", "naive"])
def test_passes_from_step_bits(gpu_available, ref_dirs2, monkeypatch, shape, method, faithful,
                               precision, solver):
    print(f"case step bits {shape} {method} {faithful} {precision} {solver}", flush=True)
    f = F.taylor_green(max(shape), noise=0.2, seed=8, shape=shape)
    fp32 = precision == "fp32"
    acc = [a.astype(np.float32).astype(np.float64) for a in f["acc"]] if fp32 else f["acc"]
    mask = (np.random.default_rng(9).random(shape) > 0.5).astype(np.float64)
    if method == "weighted":
        mask[:] = 1.0
    curl = O.curl(shape, f["delta"], acc, mask)
    thr = float(np.median(curl[curl > 0])) if method == "select" else 0.0
    m = {"plain": omni3d.PLAIN, "mask": omni3d.PLAIN_MASK, "select": omni3d.SELECT,
         "weighted": omni3d.WEIGHTED}[method]
    sv = omni3d.AFFINE if solver == "affine" else omni3d.NAIVE

    def go():
        with omni3d.Context(shape, f["delta"], density=f["rho"], method=m, threshold=thr,
                            precision=omni3d.FP32 if fp32 else omni3d.FP64, solver=sv,
                            faithful_select=faithful, max_iterations=3) as ctx:
            ctx.set_directions(ref_dirs2)
            ctx.set_field(acc, mask=None if method == "plain" else mask)
            return ctx.reconstruct()

    p, w, rep = go()
    monkeypatch.setenv("OMNI3D_MASKED", "naive")
    pn, wn, rn = go()
    assert rep.iterations == rn.iterations == 3
    unit = method in ("plain", "mask")
    if unit:
        np.testing.assert_array_equal(w, wn)
    else:
        assert F.rel_l2(w, wn) <= 1e-12
    assert F.rel_l2(p, pn) <= (1e-5 if fp32 else (1e-12 if unit else 1e-10))
