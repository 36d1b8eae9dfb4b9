"""The curl-weighted iteration in tile layout at its edges: tiles of a few
entries and of several chunks, chunks that begin inside a quad of entries, runs
of a fixed count and runs that a tolerance stops after an even or odd count
(which of the two p buffers holds the result).  Against the reference's schedule
run to the same count: weights to 1e-12, p to 1e-10 (FP64 curl quotients in
another order).
"""
import numpy as np
import pytest

import omni3d
import oracle as O
from omni3d import fields as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(3, 4, 5), (19, 18, 33), (40, 36, 44)])
# (tolerances that every shape reaches before its twelfth iteration)
@pytest.mark.parametrize("method,tol", [(omni3d.SELECT, 0.0), (omni3d.SELECT, 2e-1),
                                        (omni3d.WEIGHTED, 0.0), (omni3d.WEIGHTED, 2e-2)])
def test_curl_iteration_matches_full_passes(gpu_available, ref_dirs2, shape, method, tol):
    print(f"case curl iteration {shape} {method} {tol}", flush=True)
    f = F.taylor_green(max(shape), noise=0.1, seed=12, shape=shape)
    curl = O.curl(shape, f["delta"], f["acc"], np.ones(shape))
    thr = float(np.quantile(curl[curl > 0], 0.7)) if method == omni3d.SELECT else 0.0
    p0 = np.random.default_rng(3).normal(size=shape)

    def go(solver, iterations, tolerance):
        with omni3d.Context(shape, f["delta"], density=f["rho"], method=method, threshold=thr,
                            solver=solver, max_iterations=iterations, tolerance=tolerance) as ctx:
            ctx.set_directions(ref_dirs2)
            ctx.set_field(f["acc"], mask=np.ones(shape))
            return ctx.reconstruct(p0)

    p, w, r = go(omni3d.AFFINE, 12, tol)
    print(f"  stopped after {r.iterations}, relative change {r.rel_change:.2e}", flush=True)
    # (the relative change is over the run starts here, over every voxel in the
    # reference's schedule, so that one runs the count found here)
    q, v, s = go(omni3d.NAIVE, r.iterations, 0.0)
    assert s.iterations == r.iterations
    if tol == 0.0:
        assert r.iterations == 12
    else:
        assert r.iterations < 12 and r.rel_change < tol
        # and not a step late
        _, _, before = go(omni3d.AFFINE, r.iterations - 1, 0.0)
        assert r.iterations == 1 or before.rel_change >= tol
    assert F.rel_l2(w, v) <= 1e-12
    assert F.rel_l2(p, q) <= 1e-10
