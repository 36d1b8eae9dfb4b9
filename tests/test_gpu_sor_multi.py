"""Two red-black iterations in one pass, where a thread keeps a pair of voxels
and the columns meet: one voxel thick and two wide boxes, odd rows (a last
voxel without its pair), columns of one voxel, one more and one less than a
whole one, several parts of the planes, and an odd number of iterations (the
last alone).  Every update is the same expression on the same values as in the
half sweeps in place, so the iterates are bit-equal.
"""
import numpy as np
import pytest

import omni3d

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 2), (3, 2, 2), (1, 5, 64), (35, 15, 63), (18, 17, 65), (70, 33, 131)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("iterations", [2, 5])
def test_pairs_match_half_sweeps(gpu_available, monkeypatch, shape, iterations):
    print(f"case sor pairs {shape} {iterations}", flush=True)
    rng = np.random.default_rng(6)
    rhs = rng.normal(size=shape)
    rhs[rng.random(shape) < 0.2] = 0.0
    for start in (np.zeros(shape), rng.normal(size=shape)):
        monkeypatch.delenv("OMNI3D_SOR", raising=False)
        p, it, res = omni3d.sor_solve(rhs, p0=start, omega=1.7, max_iter=iterations, eps=0.0)
        monkeypatch.setenv("OMNI3D_SOR", "halves")
        q, jt, ref = omni3d.sor_solve(rhs, p0=start, omega=1.7, max_iter=iterations, eps=0.0)
        assert it == jt == iterations
        np.testing.assert_array_equal(p, q)
        np.testing.assert_array_equal(res, ref)
