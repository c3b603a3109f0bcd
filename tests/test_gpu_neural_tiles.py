"""The training kernel's tilings against the oracle with bf16-rounded operands
(oracle/mlp.py): one tile of 64 samples, a workgroup per CU, the first batch
on 128-sample tiles (its last tile half full), several tiles per workgroup;
the batch wraps around the training set.  Bar per tensor: 2e-3 of its norm,
as for the gradient of the 4,096-sample batch (rare one-ulp flips of the
bf16 roundings)."""
import numpy as np
import pytest

import cudasphnew_amd as S
from oracle import mlp as M

pytestmark = pytest.mark.gpu

LO, HI = np.array([-0.1, 0.0, 0.2], np.float32), np.array([0.9, 1.3, 1.0], np.float32)


@pytest.mark.parametrize("batch", [64, 16384, 16448, 40000])
def test_gradient_of_every_tiling(batch):
    rng = np.random.default_rng(batch)
    x = (LO + (HI - LO) * rng.random((5000, 3))).astype(np.float32)
    d = (0.3 * np.sin(3 * x[:, 0]) - 0.2 * x[:, 1] + 0.1).astype(np.float32)
    n = S.NeuralSDF(LO, HI, seed=5, out_scale=0.5)
    th = M.xavier_init(4).astype(np.float32)
    n.set_params(th)
    n.set_samples(np.column_stack([x, d]))
    first = 4321
    loss, g = n.gradient(first, batch)
    i = (first + np.arange(batch)) % 5000
    u = M.normalized(x[i], LO, HI)
    loss_b, g_b = M.loss_and_grad(th.astype(np.float64), u, M.target(d[i], 0.0, 0.5), bf=True)
    assert loss == pytest.approx(loss_b, rel=1e-4)
    for a, b in ((M.O_W1, M.O_B1), (M.O_B1, M.O_W2), (M.O_W2, M.O_B2), (M.O_B2, M.O_W3), (M.O_W3, M.O_B3),
                 (M.O_B3, M.O_W4), (M.O_W4, M.O_B4), (M.O_B4, M.NUM_PARAMS)):
        assert np.linalg.norm(g[a:b] - g_b[a:b]) <= 2e-3 * np.linalg.norm(g_b[a:b]), (a, b)
