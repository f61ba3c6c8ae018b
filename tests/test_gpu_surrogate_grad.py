"""Weight gradients are summed over slices of the batch (64 at most, of whole
32-row steps) and the slices added in order.  Against FP64 gradients of the same
network at the fewest rows, one slice and one step more, slices of unequal
length, and the largest batch: 2e-4 of the gradient's norm (split bf16 products:
2^-17 each, and the loss gradient itself from predictions 1e-5 off)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

H, IN = 128, 32


def _grad64(p, X, T):
    o, parts = 0, []
    for shape in ((H, IN), (H,), (H, H), (H,), (H, H), (H,), (H,), (1,)):
        n = int(np.prod(shape))
        parts.append(p[o:o + n].reshape(shape))
        o += n
    W1, b1, W2, b2, W3, b3, w4, b4 = parts
    sig = lambda z: 1.0 / (1.0 + np.exp(-z))
    ds = lambda z: sig(z) * (1.0 + z * (1.0 - sig(z)))
    Z1 = X @ W1.T + b1
    H1 = Z1 * sig(Z1)
    Z2 = H1 @ W2.T + b2
    H2 = Z2 * sig(Z2)
    Z3 = H2 @ W3.T + b3
    H3 = Z3 * sig(Z3)
    g = 2.0 * (H3 @ w4 + b4[0] - T) / len(X)
    d3 = np.outer(g, w4) * ds(Z3)
    d2 = (d3 @ W3) * ds(Z2)
    d1 = (d2 @ W2) * ds(Z1)
    return np.concatenate([(d1.T @ X).ravel(), d1.sum(0), (d2.T @ H1).ravel(), d2.sum(0), (d3.T @ H2).ravel(),
                           d3.sum(0), H3.T @ g, [g.sum()]])


@pytest.mark.parametrize("B", [32, 64, 2048, 2080, 4160, 65536])
def test_gradients(gpu, B):
    import torch
    from upcgen_amd.surrogate import Surrogate
    s = Surrogate(3)
    rng = np.random.default_rng(B)
    X = rng.uniform(-1.0, 1.0, (B, IN)).astype(np.float32)
    T = rng.normal(size=B).astype(np.float32)
    got = s.grad(0, torch.as_tensor(X, device="cuda"), torch.as_tensor(T, device="cuda")).cpu().numpy()
    want = _grad64(np.asarray(s.get_params(0), dtype=np.float64), X.astype(np.float64), T.astype(np.float64))
    assert got.shape == want.shape
    assert np.linalg.norm(got - want) <= 2e-4 * np.linalg.norm(want)
