"""The training pass at the edges of its tiles, rounds and grid (32 samples per wave, 128
per block and round, 256 blocks) against the float64 reference: loss and gradient within
1e-5 of their scale, the bound of the FP32 sums that test_mlp_gpu.py derives its check
from, and the same bits on a second run."""
import numpy as np
import pytest

from oracle import mlp_ref
from simplediffeq_hip import costmodel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 31, 33, 127, 128, 129, 1000, 128 * 256, 128 * 256 + 1, 70001])
def test_loss_grad_at_round_edges(ctx, n):
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(n)
    w = costmodel.init_params(7)
    w[384:448] = rng.uniform(-0.3, 0.3, 64)    # b1, b2, b3 at zero would hide their terms
    w[4544:4608] = rng.uniform(-0.3, 0.3, 64)
    w[4736:] = 0.2, -0.1
    x = rng.uniform(-1, 1, (n, 6)).astype(np.float32)
    y = rng.normal(0, 1, (n, 2)).astype(np.float32)
    cm = costmodel.CostModel(ctx, params=w)
    xd, yd = cm._dev(x), cm._dev(y)
    torch.cuda.synchronize()
    runs = []
    for _ in range(2):
        cm.grad.fill_(float("nan"))
        torch.cuda.synchronize()
        loss, grad = cm.loss_grad(xd, yd)
        torch.cuda.synchronize()
        runs.append((loss.item(), grad.cpu().numpy()))
    rl, rg = mlp_ref.loss_grad(w.astype(np.float64), x, y)
    assert abs(runs[0][0] - rl) < 1e-5 * max(1.0, rl)
    assert np.max(np.abs(runs[0][1] - rg)) < 1e-5 * max(1.0, np.max(np.abs(rg)))
    assert runs[0][0] == runs[1][0] and np.array_equal(runs[0][1], runs[1][1])
