"""Several gradients of one batch loss at once (is_grads_batched, vectorized jacobians): each row is the gradient
for its factor alone."""
import numpy as np
import pytest

from tests.test_gpu_batch_loss import _close, _loss

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("kind,etype", [("mechanical", "quad"), ("thermal", "quad"), ("neohooke", "tetra")])
def test_rows_are_the_single_gradients(kind, etype, dtype):
    loss, f0, u0 = _loss(kind, etype, 0.0, 3, dtype)
    factors = torch.tensor([1.0, -0.5, 3.0], dtype=dtype, device="cuda")
    for call in (lambda f, u: loss.ComputeBatchResidualNormLoss(f, u), lambda f, u: loss.ComputeBatchLoss(f, u)[0],
                 lambda f, u: loss.ComputeBatchLoss(f, u)[1][0], lambda f, u: loss.ComputeBatchLoss(f, u)[1][1]):
        f, u = f0.clone().requires_grad_(True), u0.clone().requires_grad_(True)
        rows = torch.autograd.grad(call(f, u), (f, u), grad_outputs=factors, is_grads_batched=True)
        for k, factor in enumerate(factors):
            for row, want in zip(rows, torch.autograd.grad(call(f, u), (f, u), grad_outputs=factor)):
                _close(row[k], want, dtype)


def test_vectorized_jacobian():
    loss, f0, u0 = _loss("thermal", "quad", 0.0, 2, torch.float64)

    def both(u):
        return torch.stack([loss.ComputeBatchLoss(f0, u)[0], loss.ComputeBatchResidualNormLoss(f0, u)])

    one = torch.autograd.functional.jacobian(both, u0)
    assert np.isfinite(one.cpu().numpy()).all()
    _close(torch.autograd.functional.jacobian(both, u0, vectorize=True), one, torch.float64)
