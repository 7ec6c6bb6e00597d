"""The loss gradient of batches beyond 65536 samples: a row of partial gradients, summed in
FP32, holds 256 samples however large the batch is, and the rows are summed in FP64."""
import numpy as np
import pytest

from oracle import mlp_oracle as MO

pytestmark = pytest.mark.gpu


def _setup(n, batch, seed):
    from cmdg import closure
    rng = np.random.default_rng(seed)
    table = rng.standard_normal((13, n)).astype(np.float32)
    table[10] = np.abs(table[10]) + 0.1
    table[11] = -np.abs(table[11]) - 0.1       # one sign: the samples' gradients do not cancel
    table[12] = np.abs(table[12]) + 1.0
    mlp = closure.MLPParams.random(seed=seed, y0=0.02, shift=rng.uniform(-0.1, 0.1, 10),
                                   scale=rng.uniform(0.3, 0.6, 10))
    mlp.flat[closure.OFF_W3:closure.OFF_B3] *= 0.05    # outputs inside the clamp
    mlp.flat[closure.OFF_B1:closure.OFF_W2] = rng.uniform(-0.2, 0.2, 32)
    mlp.flat[closure.OFF_B2:closure.OFF_W3] = rng.uniform(-0.2, 0.2, 32)
    return table, mlp, closure.ClosureTrainer(mlp, max_batch=batch)


@pytest.mark.parametrize("batch", [1 << 17, 1 << 20, 1 << 22])
def test_sums_keep_their_precision_as_the_batch_grows(batch):
    """A batch of sixteen samples over and over, its norm a power of two: every row of 256 has
    the same FP32 sums, and their FP64 sum scales them exactly, so every batch gives the bits
    of the batch of 65536."""
    import torch
    table, _, tr = _setup(16, batch, 3)
    T = torch.from_numpy(table).cuda()
    idx = torch.arange(batch, device="cuda") % 16
    small = tr.loss_grad(T, 1 << 16, idx, 2.0 ** -16).cpu().numpy().copy()
    large = tr.loss_grad(T, batch, idx, 1.0 / batch).cpu().numpy()
    assert np.isfinite(small).all() and np.abs(small[:1440]).min() > 0
    assert np.array_equal(small.view(np.uint32), large.view(np.uint32))


@pytest.mark.parametrize("batch", [65537, 65793, 300001])
def test_loss_gradient_of_ragged_large_batches(batch):
    import torch
    n = batch + 3
    table, mlp, tr = _setup(n, batch, batch)
    r = np.random.default_rng(batch + 1).integers(0, n, batch)
    got = tr.loss_grad(torch.from_numpy(table).cuda(), batch, torch.from_numpy(r).cuda(),
                       1.0 / batch).cpu().numpy().astype(np.float64)
    x = MO.normalise(table, mlp.shift, mlp.scale, r)
    L, ref = MO.loss_grad(mlp.flat, x, table[10, r].astype(np.float64), table[11, r].astype(np.float64),
                          table[12, r].astype(np.float64), 1.0 / batch)
    # FP32 throughout: three chained sums of at most 32 terms and sums over at most 256 samples
    # before FP64, each within its length times 6e-8
    tol = (3 * 32 + 256) * 6e-8
    assert abs(got[1440 + 1] - L) <= tol * abs(L)
    for a, b in ((0, 320), (320, 352), (352, 1376), (1376, 1408), (1408, 1440), (1440, 1441)):
        assert np.linalg.norm(got[a:b] - ref[a:b]) <= tol * np.linalg.norm(ref[a:b]), (a, b)
