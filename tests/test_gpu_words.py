"""The merged words of the source iteration at the edges of their layout:
few sources (groups of one row, groups whose rows have no entries and which
load the filling block alone), rows of many equal entries (words of 1, 2 and 4), one block per
group and several rounds per wavefront, groups of 4 and of 8 wavefronts.
Against the dense words (one entry per word, 64 rows per chunk): both round
every FP64 term to the same unit and add exactly, so p is bit-equal there.
FP32 ray sums iterate on FP32 increments (rounded to 2^-24 of themselves, a
few hundred terms a row) against FP64 values: 1e-6 as for the other layouts.
"""
import numpy as np
import pytest

import omni3d
from omni3d import fields as F

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (3, 4, 5), (2, 9, 130), (33, 34, 2), (31, 24, 40)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("chunks", ["", "4", "8"])
@pytest.mark.parametrize("precision", [omni3d.FP64, omni3d.FP32_KAHAN])
@pytest.mark.parametrize("tol", [0.0, 1e-2])
def test_words_agree_with_dense_words(gpu_available, ref_dirs2, monkeypatch, shape, chunks,
                                      precision, tol):
    print(f"case words {shape} chunks={chunks or 'auto'} precision={precision} tol={tol}",
          flush=True)
    f = F.taylor_green(max(shape), noise=0.05, seed=3, shape=shape)
    p0 = np.random.default_rng(4).normal(size=shape)
    dtype = np.float64 if precision == omni3d.FP64 else np.float32

    def go(group, init):
        if group:
            monkeypatch.setenv("OMNI3D_DENSE_GROUP", group)
        else:
            monkeypatch.delenv("OMNI3D_DENSE_GROUP", raising=False)
        with omni3d.Context(shape, f["delta"], density=f["rho"], precision=precision,
                            max_iterations=9, tolerance=tol) as ctx:
            ctx.set_directions(ref_dirs2)
            ctx.set_field([np.asarray(a, dtype=dtype) for a in f["acc"]], dtype=dtype)
            return ctx.reconstruct(init)

    for init in (None, p0):
        pd, wd, rd = go("1", init)
        pw, ww, rw = go(chunks, init)
        assert rw.iterations == rd.iterations
        np.testing.assert_array_equal(ww, wd)
        if precision == omni3d.FP64:
            np.testing.assert_array_equal(pw, pd)
        else:
            assert F.rel_l2(pw, pd) < 1e-6
