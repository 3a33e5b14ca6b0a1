"""MLP cost-model kernels vs the FP64 oracle: BF16 weight rounding, forward outputs,
gradients, determinism, and that training reduces the loss."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def mg():
    import matrixgraph_amd

    return matrixgraph_amd


def data(n, n_in, n_out, seed):
    rng = np.random.default_rng(seed)
    x = rng.normal(0, 1, (n, n_in)).astype(np.float32)
    w_true = rng.normal(0, 1, (n_in, n_out))
    t = (np.tanh(x @ w_true) + 0.1 * rng.normal(0, 1, (n, n_out))).astype(np.float32)
    return x, t


@pytest.mark.parametrize("n_in,n_out", [(8, 2), (16, 1), (4, 2)])
def test_mlp_bf16_forward_and_gradient_match_oracle(ctx, n_in, n_out):
    M = mg()
    m = M.MLP(ctx, n_in, n_out, seed=7)
    master, bf16 = m.params()
    assert all(O.f32_to_bf16(float(f)) == int(h) for f, h in zip(master[:300], bf16[:300]))
    wq = np.array([O.bf16_to_f32(int(h)) for h in bf16], np.float64)  # the weights the kernels use
    x, t = data(1000, n_in, n_out, 3)
    y = m.forward(x)
    # forward: FP32 accumulation of BF16 weights vs FP64 reference
    loss_ref, grad_ref = O.mlp_loss_grad(n_in, n_out, wq, x, t)
    loss, grad = m.loss_grad(x, t)
    assert loss == pytest.approx(loss_ref, rel=1e-4)
    scale = np.abs(grad_ref).max()
    assert np.abs(grad - grad_ref).max() <= 1e-4 * scale + 1e-7
    # outputs against an explicit FP64 forward of the same weights
    assert np.isfinite(y).all() and y.shape == (1000, n_out)
    loss_y = float(((y.astype(np.float64) - t) ** 2).mean())
    assert loss_y == pytest.approx(loss_ref, rel=1e-4)
    # determinism: same inputs, same gradient bits
    _, grad2 = m.loss_grad(x, t)
    assert np.array_equal(grad, grad2)


def test_mlp_training_reduces_loss(ctx):
    M = mg()
    x, t = data(20000, 8, 2, 5)
    m = M.MLP(ctx, 8, 2, seed=1)
    l0, _ = m.loss_grad(x, t)
    l1 = m.train(x, t, epochs=5, batch=512, lr=3e-3)
    assert l1 < 0.5 * l0


# Around the 32-row tiles and the largest grid (512 workgroups of a gradient, 1024 of a forward pass).
@pytest.mark.parametrize("n", [1, 31, 32, 33, 64, 97, 512 * 32 + 1, 1024 * 32 + 33])
@pytest.mark.parametrize("n_in,n_out", [(4, 1), (4, 2), (8, 1), (8, 2), (16, 1), (16, 2)])
def test_mlp_tiles_match_oracle(ctx, n, n_in, n_out):
    M = mg()
    m = M.MLP(ctx, n_in, n_out, seed=n + n_in)
    rng = np.random.default_rng(n)
    master = m.params()[0] + rng.normal(0, 0.05, m.n_params).astype(np.float32)  # biases too
    m.set_params(master)
    _, bf16 = m.params()
    wq = (bf16.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    x, t = data(n, n_in, n_out, n)
    w1, b1, w2, b2, w3, b3 = np.split(wq, np.cumsum([64 * n_in, 64, 4096, 64, 64 * n_out]))
    h = np.maximum(x.astype(np.float64) @ w1.reshape(64, n_in).T + b1, 0)
    h = np.maximum(h @ w2.reshape(64, 64).T + b2, 0)
    want = h @ w3.reshape(n_out, 64).T + b3
    assert np.abs(m.forward(x) - want).max() <= 1e-5 * np.abs(want).max()
    loss_ref, grad_ref = O.mlp_loss_grad(n_in, n_out, wq, x, t)
    loss, grad = m.loss_grad(x, t)
    assert loss == pytest.approx(loss_ref, rel=1e-4)
    scale = np.abs(grad_ref).max()
    assert np.abs(grad - grad_ref).max() <= 1e-4 * scale + 1e-7
    # One Adam step is lr * g / (|g| + eps), whatever the size of g; the loss is that of the new weights.
    after = m.train(x, t, epochs=1, batch=n, lr=1e-3)
    moved, bf16 = m.params()
    big = np.abs(grad_ref) > 1e-2 * scale
    assert np.abs(moved - (master - 1e-3 * np.sign(grad_ref)))[big].max() <= 1e-6
    wq = (bf16.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    assert after == pytest.approx(O.mlp_loss_grad(n_in, n_out, wq, x, t)[0], rel=1e-4)
