"""The walks over a tile by 16-bit positions, where the positions and edges end:
one whole tile, one voxel more than a tile in an axis (edges that lead into and
out of tiles of one voxel), thin grids, 8^3 and 16^3 tiles.  The forward passes
against the engine with one lane per ray (FP64 sums of the same terms: 1e-12;
FP32 ray sums 1e-5), the transposed ones against the full-volume walks with one
lane per ray (1e-12).
"""
import numpy as np
import pytest

import omni3d
from omni3d import fields as F

pytestmark = pytest.mark.gpu

SHAPES = [(16, 16, 16), (17, 16, 33), (8, 9, 16), (2, 3, 50)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("bits", [3, 4])
@pytest.mark.parametrize("precision", [omni3d.FP64, omni3d.FP32_KAHAN])
def test_forward_walks(gpu_available, ref_dirs2, monkeypatch, shape, bits, precision):
    print(f"case tile walk {shape} {bits} {precision}", flush=True)
    f = F.taylor_green(max(shape), noise=0.1, seed=4, shape=shape)
    dtype = np.float64 if precision == omni3d.FP64 else np.float32

    def go():
        with omni3d.Context(shape, f["delta"], density=f["rho"], precision=precision,
                            max_iterations=3) as ctx:
            ctx.set_tile_shape(bits, 256)
            ctx.set_directions(ref_dirs2)
            ctx.set_field([np.asarray(a, dtype=dtype) for a in f["acc"]], dtype=dtype)
            return ctx.reconstruct()

    p, w, _ = go()
    monkeypatch.setenv("OMNI3D_ENGINE", "rays")
    q, v, _ = go()
    np.testing.assert_array_equal(w, v)
    assert F.rel_l2(p, q) <= (1e-12 if precision == omni3d.FP64 else 1e-5)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("bits", [3, 4])
def test_transposed_walks(gpu_available, ref_dirs2, shape, bits):
    import torch
    print(f"case transposed tile walk {shape} {bits}", flush=True)
    V = int(np.prod(shape))
    gen = torch.Generator(device="cuda").manual_seed(5)
    y = torch.randn(V, dtype=torch.float64, device="cuda", generator=gen)
    out = []
    for solver in (omni3d.AFFINE, omni3d.NAIVE):
        with omni3d.Context(shape, (0.1, 0.2, 0.3), max_iterations=3, solver=solver) as ctx:
            ctx.set_tile_shape(bits, 1024)
            ctx.set_directions(ref_dirs2)
            ctx.set_field([np.zeros(shape)] * 3)
            dg = torch.empty(3 * V, dtype=torch.float64, device="cuda")
            ctx.backward_device(y.data_ptr(), dg.data_ptr())
            torch.cuda.synchronize()
            out.append(dg)
    assert float(torch.linalg.norm(out[1])) > 0
    assert float(torch.linalg.norm(out[0] - out[1]) / torch.linalg.norm(out[1])) < 1e-12
