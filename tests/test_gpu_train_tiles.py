"""The loss gradient at the edges of its tiles: 16 samples a wave, four waves a workgroup, a
row of partial gradients for every 64 samples up to 256 rows, then several tiles a wave."""
import numpy as np
import pytest

from oracle import mlp_oracle as MO

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 15, 16, 17, 63, 64, 65, 129, 16383, 16384, 16385, 16448, 40001])
@pytest.mark.parametrize("rows", ["in order", "drawn"])
def test_loss_gradient_tile_edges(batch, rows):
    import torch
    from cmdg import closure
    rng = np.random.default_rng(batch)
    n = batch + 3
    table = rng.standard_normal((13, n)).astype(np.float32)
    table[10] = np.abs(table[10]) + 0.1
    table[11] = -np.abs(table[11]) - 0.1       # one sign: the samples' gradients do not cancel
    table[12] = np.abs(table[12]) + 1.0
    mlp = closure.MLPParams.random(seed=batch, y0=0.02, shift=rng.uniform(-0.1, 0.1, 10),
                                   scale=rng.uniform(0.3, 0.6, 10))
    mlp.flat[closure.OFF_W3:closure.OFF_B3] *= 0.05    # outputs inside the clamp
    mlp.flat[closure.OFF_B1:closure.OFF_W2] = rng.uniform(-0.2, 0.2, 32)
    mlp.flat[closure.OFF_B2:closure.OFF_W3] = rng.uniform(-0.2, 0.2, 32)
    tr = closure.ClosureTrainer(mlp, max_batch=batch)
    idx = None if rows == "in order" else torch.from_numpy(rng.integers(0, n, batch)).cuda()
    got = tr.loss_grad(torch.from_numpy(table).cuda(), batch, idx, 1.0 / batch).cpu().numpy().astype(np.float64)
    r = np.arange(batch) if idx is None else idx.cpu().numpy()
    x = MO.normalise(table, mlp.shift, mlp.scale, r)
    L, ref = MO.loss_grad(mlp.flat, x, table[10, r].astype(np.float64), table[11, r].astype(np.float64),
                          table[12, r].astype(np.float64), 1.0 / batch)
    # FP32 throughout: three chained sums of at most 32 terms and sums over samples at most 128
    # terms long before FP64, each within its length times 6e-8
    tol = (3 * 32 + 128) * 6e-8
    assert abs(got[1440 + 1] - L) <= tol * abs(L)
    for a, b in ((0, 320), (320, 352), (352, 1376), (1376, 1408), (1408, 1440), (1440, 1441)):
        assert np.linalg.norm(got[a:b] - ref[a:b]) <= tol * np.linalg.norm(ref[a:b]), (a, b)
