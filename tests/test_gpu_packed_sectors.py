"""Packed save_everystep rows written by 64-byte sectors of the output: output buffers that
begin anywhere in a sector (on a whole element, and off it, where rows are written one by one),
trajectories of two rows and of many, both precisions and states of 1 to 8 components: the rows
of an aligned buffer, and nothing written before the buffer or after the last row."""
import numpy as np
import pytest

from helpers import bits_equal
from simplediffeq_hip import _abi, runtime
from test_gpu_packed_runs import _rhs

pytestmark = pytest.mark.gpu


def _solve(c, n, n_state, dtype, span, shift, rows):
    import torch
    rhs, n_param = _rhs(c, n_state)
    rng = np.random.default_rng(n_state)
    u0 = rng.uniform(-1.0, 1.0, (n_state, n))
    p = rng.uniform(0.5, 3.0, (n_param, n))
    ts = np.zeros((2, n))
    ts[1] = rng.permutation(np.linspace(0.0, span, n))
    d = runtime.make_desc(_abi.ALG_ATSIT5, rhs=rhs, n_traj=n, dt=0.1, abstol=1e-6, reltol=1e-4,
                          dtype=dtype, save_everystep=True, save_layout=_abi.SAVE_PACKED)
    b = runtime.EnsembleBuffers(d, n_state, u0, p, tspan=ts, backend="torch", device="cuda:0",
                                steps_capacity=rows)
    su, st = shift  # bytes
    es = 8 if dtype == _abi.F64 else 4
    u = torch.zeros(rows * n_state * es + 192, dtype=torch.uint8, device="cuda:0")
    t = torch.zeros(rows * 8 + 192, dtype=torch.uint8, device="cuda:0")
    u.fill_(0xa5)
    t.fill_(0xa5)
    b.io.u_steps = u.data_ptr() + 64 + su
    b.io.t_steps = t.data_ptr() + 64 + st
    torch.cuda.synchronize()
    assert c.solve(d, b) == 0
    assert c.stats()["schedule"] == _abi.SCHED_ONE_LAUNCH
    used = int(b.numpy("steps_offset")[n])
    out = []
    for buf, s, width in ((u, su, n_state * es), (t, st, 8)):
        h = buf.cpu().numpy()
        assert (h[:64 + s] == 0xa5).all() and (h[64 + s + used * width:] == 0xa5).all()
        out.append(h[64 + s:64 + s + used * width].copy())
    return out, used


@pytest.mark.parametrize("n_state,dtype,span", [
    (3, _abi.F64, 0.05), (3, _abi.F64, 0.8), (1, _abi.F64, 0.8), (4, _abi.F64, 0.8),
    (3, _abi.F32, 0.8), (1, _abi.F32, 0.05), (8, _abi.F32, 0.8)])
def test_rows_anywhere_in_a_sector(n_state, dtype, span):
    c = runtime.Context(0)
    n = 600_001
    es = 8 if dtype == _abi.F64 else 4
    ref, rows = _solve(c, n, n_state, dtype, span, (0, 0), n * 24)
    for shift in ((es, 56), (3 * es, 8), (64 - es, 24), (4 if es == 8 else 0, 4)):
        got, used = _solve(c, n, n_state, dtype, span, shift, rows)
        assert used == rows
        assert bits_equal(got[0], ref[0]) and bits_equal(got[1], ref[1]), shift
    c.close()
