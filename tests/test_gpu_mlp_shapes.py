"""The network's matrix-core kernels at the edges of their tiles: layer widths
around the 16, 32, 64 and 256-wide blocks, batches around the row tiles and
the batch slices, against the FP64 reference with the same BF16 rounding."""
import numpy as np
import pytest

from mopac_gpu_amd import guess
from oracle import mlp_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", ([1, 1], [3, 5, 2], [31, 33, 16], [96, 256, 256, 16], [168, 65, 257, 20],
                                  [300, 64, 7]))
@pytest.mark.parametrize("batch", (1, 15, 17, 129, 300))
def test_forward_and_gradients(dims, batch):
    rng = np.random.Generator(np.random.PCG64(batch + len(dims)))
    params = guess.init_params(5, dims)
    params += 0.05 * rng.standard_normal(params.size).astype(np.float32)
    x = rng.standard_normal((batch, dims[0])).astype(np.float32)
    t = rng.standard_normal((batch, dims[-1])).astype(np.float32)
    m = guess.MLP(params, dims=dims)
    try:
        y = m.forward(x)
        g, loss = m.gradients(x, t)
    finally:
        m.close()
    y_ref = mlp_ref.forward(params, dims, x)[-1]
    loss_ref, g_ref = mlp_ref.loss_and_grad(params, dims, x, t)
    # a hidden activation whose FP32 sum rounds to the other BF16 neighbour
    # (one part in 2^8) reaches an output through one of its layer's weights:
    # a few of them at the narrowest layers bound both errors
    assert np.linalg.norm(y - y_ref) <= 2.0 ** -8 * np.linalg.norm(y_ref) + 1e-6
    assert abs(loss - loss_ref) <= 2.0 ** -8 * loss_ref
    assert np.linalg.norm(g - g_ref) <= 2.0 ** -7 * np.linalg.norm(g_ref)


def test_gradient_keeps_fp32_operands():
    """One linear layer: dW is X^T dZ with X exact in BF16 and dZ in FP32, so
    nothing but the FP32 sums (a batch of terms, in slices of at most 128) is
    rounded.  A dZ rounded to BF16 would be off by 2^-9 a term."""
    batch, dims = 512, [64, 64]
    rng = np.random.Generator(np.random.PCG64(3))
    x = rng.integers(-128, 129, (batch, 64)).astype(np.float32) / 16.0
    t = rng.standard_normal((batch, 64)).astype(np.float32)
    params = np.zeros(64 * 64 + 64, dtype=np.float32)
    m = guess.MLP(params, dims=dims)
    try:
        g, _ = m.gradients(x, t)
    finally:
        m.close()
    dz = -2.0 * t.astype(np.float64) / t.size
    want = x.astype(np.float64).T @ dz
    terms = np.abs(x.astype(np.float64)).T @ np.abs(dz)
    eps = np.finfo(np.float32).eps
    assert np.all(np.abs(g[:64 * 64].reshape(64, 64) - want) <= 0.5 * np.sqrt(batch) * eps * terms)
    assert np.all(np.abs(g[64 * 64:] - dz.sum(0)) <= 0.5 * np.sqrt(batch) * eps * np.abs(dz).sum(0))
