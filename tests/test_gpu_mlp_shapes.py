"""GPU: the order model at the sizes where its kernels change (rows per block,
sample slices and their remainders, other input widths, other hidden widths),
against the oracle's float64 forward and gradients.  Tolerance: fp32 sums of up
to 272 products of magnitude near 1 are within 1e-5 of the result's scale; a
unit whose sum is that near zero may be active on one side only, which moves
the gradient by one sample's share."""
import numpy as np
import pytest

from gem_amd.learned import OrderModel
from oracle import mlp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,width,hidden", [(1, 272, 128), (7, 272, 128), (8, 272, 128), (65, 272, 128),
                                            (2048, 272, 128), (2049, 272, 128), (8225, 272, 128), (70, 16, 128),
                                            (2500, 144, 128), (40, 20, 128), (40, 272, 64)])
def test_forward_and_gradient(gpu_ctx, n, width, hidden):
    rng = np.random.default_rng(n + width)
    feats = rng.integers(0, 500, size=(n, width)).astype(np.int32)
    targets = rng.uniform(-2, 2, n).astype(np.float32)
    model = OrderModel(gpu_ctx, seed=n, in_dim=width, hidden=hidden)
    p = model.get_params() + rng.uniform(-0.02, 0.02, model.num_params).astype(np.float32)
    model.set_params(p)
    _, _, _, y, _ = mlp.forward(p, feats, width, hidden)
    assert np.max(np.abs(model.predict(feats) - y)) <= 1e-5 * max(1.0, np.abs(y).max())
    loss, grad = model.loss_grad(feats, targets)
    ref_loss, ref = mlp.loss_grad(p, feats, targets, width, hidden)
    assert abs(loss - ref_loss) <= 1e-5 * abs(ref_loss)
    assert np.linalg.norm(grad - ref) <= (1e-5 + 1.0 / n / 100) * np.linalg.norm(ref)
    model.close()
