"""Device memory passed on from released objects: contexts made, run and
dropped by two threads at once, each on a stream of its own, give bit for bit
what they give alone (a block still in use by the other stream must not
serve), whatever sizes were released before; and what waits is bounded and
returned on request.
"""
import ctypes
import threading

import numpy as np
import pytest
import torch

import omni3d
from omni3d import fields as F

pytestmark = pytest.mark.gpu

SHAPES = [(24, 20, 28), (9, 40, 17), (33, 30, 31)]


def _run(shape, dirs, stream, method):
    f = F.taylor_green(max(shape), noise=0.05, seed=2, shape=shape)
    with omni3d.Context(shape, f["delta"], density=f["rho"], method=method,
                        max_iterations=6) as ctx:
        assert omni3d.lib().omni3d_set_stream(ctx._h, ctypes.c_void_p(stream.cuda_stream)) == 0
        ctx.set_directions(dirs)
        ctx.set_field(f["acc"], mask=None if method == omni3d.PLAIN else np.ones(shape))
        p, w, _ = ctx.reconstruct()
    return p, w


def test_threads_share_released_memory(gpu_available, ref_dirs2):
    jobs = [(s, m) for s in SHAPES for m in (omni3d.PLAIN, omni3d.PLAIN_MASK)]
    alone = {}
    for j in jobs:
        print(f"case pool alone {j}", flush=True)
        alone[j] = _run(j[0], ref_dirs2, torch.cuda.Stream(), j[1])
    bad, errors = [], []

    def work(order):
        try:
            st = torch.cuda.Stream()
            for j in order:
                p, w = _run(j[0], ref_dirs2, st, j[1])
                if not (np.array_equal(p, alone[j][0]) and np.array_equal(w, alone[j][1])):
                    bad.append(j)
        except Exception as e:  # (reported by the main thread)
            errors.append(e)

    print("case pool two threads", flush=True)
    t = [threading.Thread(target=work, args=(jobs * 3,)),
         threading.Thread(target=work, args=(jobs[::-1] * 3,))]
    for x in t:
        x.start()
    for x in t:
        x.join()
    assert not errors and not bad


def test_released_memory_is_returned(gpu_available, ref_dirs2):
    print("case pool returned", flush=True)
    L = omni3d.lib()
    L.omni3d_dropin_release()
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    _run(SHAPES[2], ref_dirs2, torch.cuda.Stream(), omni3d.PLAIN)
    torch.cuda.synchronize()
    assert before - torch.cuda.mem_get_info()[0] <= (2 << 30) + (64 << 20)
    L.omni3d_dropin_release()
    torch.cuda.synchronize()
    # (a stream's and the graph's own memory may stay: 64 MiB)
    assert before - torch.cuda.mem_get_info()[0] <= 64 << 20
