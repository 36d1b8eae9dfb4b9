"""Tile passes whose tiles are dealt to several workgroups, at the edges of
the rule: one tile with fewer segments than its 16 workgroups have threads
(empty parts), thin remainder tiles, and enough tiles that each is one
workgroup's again.  Against the FP64 oracle (kernel.cu:8805-8861); the sums
are the same terms in another order, so the bars are those of the one-
workgroup passes: p <= 1e-12 (1e-10 with curl weights, whose quotients
amplify the order), counts exact, FP32 ray sums <= 1e-5.
"""
import numpy as np
import pytest

import omni3d
import oracle as O
from omni3d import fields as F

pytestmark = pytest.mark.gpu

# (shape, tile bits): 1, 6, 12 and 512 tiles
CASES = [((3, 4, 5), 4), ((33, 16, 17), 4), ((20, 37, 18), 4), ((64, 64, 64), 3)]


def _field(shape, seed=5):
    f = F.taylor_green(max(shape), noise=0.05, seed=seed, shape=shape)
    rng = np.random.default_rng(seed)
    f["mask"] = (rng.random(shape) > 0.1).astype(np.float64)
    return f


@pytest.mark.parametrize("shape,bits", CASES)
@pytest.mark.parametrize("method", ["plain", "mask", "select", "weighted"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_tile_parts(gpu_available, ref_dirs2, shape, bits, method, precision):
    print(f"case tile parts {shape} {bits} {method} {precision}", flush=True)
    f = _field(shape)
    m = {"plain": (omni3d.PLAIN, O.PLAIN), "mask": (omni3d.PLAIN_MASK, O.PLAIN_MASK),
         "select": (omni3d.SELECT, O.SELECT), "weighted": (omni3d.WEIGHTED, O.WEIGHTED)}[method]
    fp32 = precision == "fp32"
    acc = [a.astype(np.float32).astype(np.float64) for a in f["acc"]] if fp32 else f["acc"]
    curl = f["mask"] if method == "mask" else O.curl(shape, f["delta"], acc, f["mask"])
    thr = float(np.quantile(curl[curl > 0], 0.8)) if method == "select" else 0.0
    iters = 2 if shape == (64, 64, 64) else 4
    with omni3d.Context(shape, f["delta"], density=f["rho"], method=m[0], threshold=thr,
                        precision=omni3d.FP32 if fp32 else omni3d.FP64,
                        max_iterations=iters) as ctx:
        ctx.set_tile_shape(bits, 1024)
        ctx.set_directions(ref_dirs2)
        ctx.set_field(acc, mask=None if method == "plain" else f["mask"])
        p, w, rep = ctx.reconstruct()
    po, co, it, _ = O.reconstruct(shape, ref_dirs2, 1.0, f["delta"], f["rho"], acc,
                                  curl=None if method == "plain" else curl, threshold=thr,
                                  method=m[1], max_iter=iters)
    assert rep.iterations == it
    unit = method in ("plain", "mask")
    if unit:
        assert np.array_equal(w, co)
    else:
        assert F.rel_l2(w, co) <= 1e-12
    assert F.rel_l2(p, po) <= (1e-5 if fp32 else (1e-12 if unit else 1e-10))


@pytest.mark.parametrize("shape,bits", CASES)
def test_adjoint_tile_parts(gpu_available, ref_dirs2, shape, bits):
    """<F g, y> = <g, F^T y> in FP64: both sides sum V terms, so the bar is
    the transpose identity's of the one-workgroup passes, 1e-12."""
    import torch
    print(f"case adjoint tile parts {shape} {bits}", flush=True)
    V = int(np.prod(shape))
    gen = torch.Generator(device="cuda").manual_seed(3)
    g = torch.randn(3 * V, device="cuda", dtype=torch.float64, generator=gen)
    y = torch.randn(V, device="cuda", dtype=torch.float64, generator=gen)
    p, dg = torch.empty_like(y), torch.empty_like(g)
    with omni3d.Context(shape, (0.1, 0.2, 0.15), max_iterations=3) as ctx:
        ctx.set_tile_shape(bits, 1024)
        ctx.set_directions(ref_dirs2)
        ctx.forward_device(g.data_ptr(), p.data_ptr())
        ctx.backward_device(y.data_ptr(), dg.data_ptr())
    torch.cuda.synchronize()
    lhs, rhs = float(p @ y), float(g @ dg)
    assert abs(lhs - rhs) <= 1e-12 * float(p.norm() * y.norm())
