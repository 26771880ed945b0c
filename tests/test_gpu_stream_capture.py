"""A solve that the caller captures into a graph of their own, on a context that has no
scratch yet: the schedules and layouts that the library would choose by size keep parked
records or rows in the context's scratch, which cannot be allocated during a capture and which
a later, larger solve frees, so a captured solve does without them.  Every replay, also after
such a solve, gives the eager solve's bits."""
import numpy as np
import pytest

from helpers import bits_equal
from simplediffeq_hip import _abi, inputs, runtime

pytestmark = pytest.mark.gpu

FIELDS = ("u_end", "t_end", "retcode", "naccept", "nreject")


def _bufs(n, seed, span=0.5):
    u0, p = inputs.lorenz_wide(n, seed=seed)
    d = runtime.make_desc(_abi.ALG_ATSIT5, n_traj=n, tspan=(0.0, span), dt=0.1, abstol=1e-6,
                          reltol=1e-5)
    return d, runtime.EnsembleBuffers(d, 3, u0, p, backend="torch", device="cuda:0")


def test_replays_of_a_captured_solve():
    import torch
    n = 400_001  # beyond what fits the GPU at once
    ref_ctx = runtime.Context(0)
    d, ref = _bufs(n, 3)
    ref_ctx.solve(d, ref)
    assert ref_ctx.stats()["schedule"] == _abi.SCHED_STAGED
    ref_ctx.close()

    c = runtime.Context(0)
    d, b = _bufs(n, 3)
    later = [_bufs(m, 4) for m in (500_003, 900_001)]
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        c.solve(d, b, sync=False)
    assert c.stats()["schedule"] == _abi.SCHED_PERSISTENT
    for k in range(3):
        b.u_end.zero_()
        b.naccept.zero_()
        g.replay()
        torch.cuda.synchronize()
        for f in FIELDS:
            assert bits_equal(b.numpy(f), ref.numpy(f)), (k, f)
        if k < 2:  # the context's scratch is allocated, then replaced by a larger one
            c.solve(*later[k])
            assert c.stats()["schedule"] == _abi.SCHED_STAGED
            assert (later[k][1].numpy("retcode") == 0).all()
    c.close()
