"""The learned cost model's network: the FP64 oracle pinned by central
differences and a closed-form network (CPU), then libfot's MFMA GEMM,
forward, gradients and training against the oracle (gpu)."""
import numpy as np
import pytest

import mlp_oracle as MO


def _rand_problem(rng, rows, n_in, hidden, n_out, masked=True):
    p = rng.normal(0, 0.5, hidden * n_in + hidden + hidden * hidden + hidden + n_out * hidden
                   + n_out)
    x = rng.normal(0, 1, (rows, n_in))
    t = rng.normal(0, 1, (rows, n_out))
    m = (rng.random((rows, n_out)) > 0.2).astype(np.float64) if masked else None
    return p, x, t, m


def test_oracle_gradient_matches_central_differences():
    rng = np.random.default_rng(0)
    n_in, hidden, n_out = 5, 7, 3
    p, x, t, m = _rand_problem(rng, 20, n_in, hidden, n_out)
    _, g = MO.loss_grad(p, x, t, m, n_in, hidden, n_out)
    idx = rng.choice(p.size, 60, replace=False)
    num = MO.numeric_grad(p, x, t, m, n_in, hidden, n_out, idx)
    np.testing.assert_allclose(g[idx], num, rtol=1e-5, atol=1e-8)


def test_oracle_forward_closed_form():
    # W1 = [I; -I], W2 = I, W3 = [I, -I]: relu(x) - relu(-x) = x exactly
    n = 4
    W1 = np.vstack([np.eye(n), -np.eye(n)])
    W2 = np.eye(2 * n)
    W3 = np.hstack([np.eye(n), -np.eye(n)])
    p = np.concatenate([W1.ravel(), np.zeros(2 * n), W2.ravel(), np.zeros(2 * n), W3.ravel(),
                        np.zeros(n)])
    x = np.random.default_rng(1).normal(size=(9, n))
    y, _ = MO.forward(p, x, n, 2 * n, n)
    np.testing.assert_array_equal(y, x)


# ---- GPU ------------------------------------------------------------------
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,ta,tb", [(1, 1, 1, False, False), (17, 5, 3, False, False),
                                         (64, 64, 24, False, True), (100, 6, 64, False, True),
                                         (6, 64, 100, True, False), (33, 70, 19, True, True),
                                         (257, 64, 64, False, True)])
def test_gemm_mfma_matches_numpy(gpu, M, N, K, ta, tb):
    from cuda_fot_amd.mlp import gemm
    rng = np.random.default_rng(M * 1000 + N * 10 + K)
    a = rng.normal(size=(K, M) if ta else (M, K)).astype(np.float32)
    b = rng.normal(size=(N, K) if tb else (K, N)).astype(np.float32)
    A = a.T.astype(np.float64) if ta else a.astype(np.float64)
    B = b.T.astype(np.float64) if tb else b.astype(np.float64)
    ref = A @ B
    scale = np.abs(A) @ np.abs(B)
    c = gemm(a, b, ta, tb)
    assert c.shape == (M, N)
    assert np.all(np.abs(c - ref) <= 2e-6 * scale + 1e-30), np.abs(c - ref).max()


@pytest.mark.gpu
def test_mlp_forward_and_gradient_match_oracle(gpu):
    from cuda_fot_amd.mlp import MLP
    rng = np.random.default_rng(3)
    net = MLP(24, 64, 6, seed=5)
    p = net.get_params().astype(np.float64)
    x = rng.normal(size=(333, 24)).astype(np.float32)
    t = rng.normal(size=(333, 6)).astype(np.float32)
    m = (rng.random((333, 6)) > 0.3).astype(np.float32)
    y = net.forward(x)
    yr, _ = MO.forward(p, x, 24, 64, 6)
    np.testing.assert_allclose(y, yr, rtol=1e-4, atol=1e-4 * np.abs(yr).max())
    loss, g = net.loss_grad(x, t, m)
    lr, gr = MO.loss_grad(p, x, t, m, 24, 64, 6)
    assert abs(loss - lr) <= 1e-4 * lr
    # per parameter block, relative to the block's largest gradient
    k = 0
    for shape in [(64, 24), (64,), (64, 64), (64,), (6, 64), (6,)]:
        n = int(np.prod(shape))
        gb, rb = g[k:k + n], gr[k:k + n]
        np.testing.assert_allclose(gb, rb, atol=2e-4 * np.abs(rb).max() + 1e-12, rtol=0)
        k += n


@pytest.mark.gpu
def test_mlp_training_fits_a_smooth_target(gpu):
    from cuda_fot_amd.mlp import MLP
    rng = np.random.default_rng(4)
    x = rng.normal(size=(512, 24)).astype(np.float32)
    t = np.stack([np.sin(x[:, i]) + 0.5 * x[:, i + 6] for i in range(6)], 1).astype(np.float32)
    net = MLP(24, 64, 6, seed=1)
    losses = net.train(x, t, epochs=600, lr=3e-3)
    assert losses[-1] < 0.1 * losses[0], (losses[0], losses[-1])
    # the trained parameters reproduce the reported loss through the oracle
    lr_, _ = MO.loss_grad(net.get_params().astype(np.float64), x, t, None, 24, 64, 6)
    assert lr_ < 0.1 * losses[0]


@pytest.mark.gpu
@pytest.mark.parametrize("n_in,hidden,n_out,rows,masked", [
    (1, 1, 1, 1, False), (24, 64, 6, 16, True), (24, 64, 6, 17, False), (33, 40, 7, 95, True),
    (64, 64, 16, 4096, True), (24, 64, 6, 4113, True), (32, 5, 16, 300, False),
    (24, 65, 6, 50, True), (65, 16, 3, 50, False), (8, 16, 17, 50, True)])
def test_mlp_step_at_tile_edges(gpu, n_in, hidden, n_out, rows, masked):
    """Gradient and a step of training at the edges of the one-workgroup
    network's tiles (rows of 16, widths of 32 and 64, 16 outputs, more rows
    than workgroups take at once) and just beyond, where the layers run one
    by one."""
    from cuda_fot_amd.mlp import MLP
    rng = np.random.default_rng(n_in * 1000 + rows)
    net = MLP(n_in, hidden, n_out, seed=5)
    p = net.get_params().astype(np.float64)
    x = rng.normal(size=(rows, n_in)).astype(np.float32)
    t = rng.normal(size=(rows, n_out)).astype(np.float32)
    m = (rng.random((rows, n_out)) > 0.2).astype(np.float32) if masked else None
    loss, g = net.loss_grad(x, t, m)
    lr, gr = MO.loss_grad(p, x, t, m, n_in, hidden, n_out)
    assert abs(loss - lr) <= 1e-5 * lr
    k = 0
    for shape in [(hidden, n_in), (hidden,), (hidden, hidden), (hidden,), (n_out, hidden),
                  (n_out,)]:
        n = int(np.prod(shape))
        # FP32 sums of up to 4113 rows: 4113 * 2^-24 = 2.5e-4 of the sum of
        # magnitudes at worst
        np.testing.assert_allclose(g[k:k + n], gr[k:k + n],
                                   atol=2.5e-4 * np.abs(gr[k:k + n]).max() + 1e-12, rtol=0)
        k += n
    losses = net.train(x, t, m, epochs=3, lr=1e-3, weight_decay=0.1)
    assert losses[0] == loss
    # Adam's first steps move a parameter by at most about lr each, along its
    # gradient's sign where that is not lost in rounding
    step = net.get_params() - p
    assert np.all(np.abs(step) <= 3.1e-3)
    sure = np.abs(gr + 0.1 * p) > 0.2 * np.abs(gr + 0.1 * p).max()
    assert np.all(step[sure] * (gr + 0.1 * p)[sure] < 0)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [15, 16, 17, 31])
def test_mlp_step_rows_past_the_end_stay_out(gpu, rows):
    """Weights with which an input of zeros overflows the second layer and the
    given rows do not: the rows that fill up the last tile add nothing."""
    from cuda_fot_amd.mlp import MLP
    n_in, hidden, n_out = 3, 20, 5
    net = MLP(n_in, hidden, n_out, seed=1)
    p = net.get_params()
    w1, b1 = hidden * n_in, hidden
    p[:w1] = -1e30 / n_in       # with x = 1: exactly cancelled by the bias or below
    p[w1:w1 + b1] = 0.9e30
    p[w1 + b1:w1 + b1 + hidden * hidden] = 1e12
    p[w1 + b1 + hidden * hidden:w1 + b1 + hidden * hidden + hidden] = 0.5
    net.set_params(p)
    x = np.ones((rows, n_in), np.float32)
    t = np.random.default_rng(rows).normal(size=(rows, n_out)).astype(np.float32)
    loss, g = net.loss_grad(x, t, None)
    lr, gr = MO.loss_grad(p.astype(np.float64), x, t, None, n_in, hidden, n_out)
    assert np.isfinite(g).all() and abs(loss - lr) <= 1e-5 * lr
    # FP32 sums of up to 31 rows and 20 units: 64 roundings of the terms'
    # magnitudes, which weights and hidden values below 1 scale down
    y, _ = MO.forward(p.astype(np.float64), x, n_in, hidden, n_out)
    np.testing.assert_allclose(g, gr, atol=64 * 2.0 ** -24 * 2 * np.abs(y - t).mean(), rtol=0)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [256, 4096 * 3, 4096 * 11, 4096 * 37 + 256])
def test_mlp_loss_of_equal_terms_is_the_term(gpu, rows):
    """Every output misses its target by the same value: the mean of equal FP32
    terms is the term, to the last bit, however many are summed."""
    from cuda_fot_amd.mlp import MLP
    net = MLP(1, 1, 1)
    net.set_params(np.zeros(net.num_params, np.float32))
    for value in np.float32([0.1, 1.7, 3.3333]):
        loss, _ = net.loss_grad(np.ones((rows, 1), np.float32), np.full((rows, 1), value),
                                None)
        assert np.float32(loss) == value * value


def _adam(p, x, t, mask, shape, epochs, lr, decay, state, noise=None):
    """FP64 Adam on the oracle's gradient; state: moments and steps taken.  noise
    (a generator): the gradients off by 16 FP32 roundings of the largest."""
    b1, b2, eps = (float(np.float32(v)) for v in (0.9, 0.999, 1e-8))
    losses = []
    for _ in range(epochs):
        loss, g = MO.loss_grad(p, x, t, mask, *shape)
        losses.append(loss)
        if noise is not None:
            g = g + 16 * 2.0 ** -24 * np.abs(g).max() * noise.standard_normal(g.size)
        g = g + decay * p
        state["n"] += 1
        state["m"] = b1 * state["m"] + (1 - b1) * g
        state["v"] = b2 * state["v"] + (1 - b2) * g * g
        rate = lr * np.sqrt(1 - b2 ** state["n"]) / (1 - b1 ** state["n"])
        p = p - rate * state["m"] / (np.sqrt(state["v"]) + eps)
    return p, losses


@pytest.mark.gpu
@pytest.mark.parametrize("n_in,hidden,n_out,rows,masked", [
    (24, 64, 6, 95, True), (33, 40, 7, 200, False),  # in two launches
    (24, 65, 6, 50, True), (65, 16, 3, 50, False)])  # layer by layer
def test_mlp_training_follows_adam(gpu, n_in, hidden, n_out, rows, masked):
    """Losses and parameters over two calls of train() against FP64 Adam: within
    ten times what gradients off by 16 FP32 roundings change in it.  (A decay rate
    of 0.998 for 0.999 moves the median parameter 50 times as far.)"""
    from cuda_fot_amd.mlp import MLP
    rng = np.random.default_rng(rows)
    net = MLP(n_in, hidden, n_out)
    net.set_params(rng.normal(0, 0.2, net.num_params).astype(np.float32))
    p0 = net.get_params().astype(np.float64)
    x = rng.normal(size=(rows, n_in)).astype(np.float32)
    t = rng.normal(size=(rows, n_out)).astype(np.float32)
    m = (rng.random((rows, n_out)) > 0.2).astype(np.float32) if masked else None
    calls = ((6, float(np.float32(0.02))), (4, float(np.float32(0.01))))
    decay = float(np.float32(0.1))
    runs = []
    for noise in (None, np.random.default_rng(1)):
        state, p, losses = dict(m=0.0, v=0.0, n=0), p0, []
        for epochs, lr in calls:
            p, l = _adam(p, x, t, m, (n_in, hidden, n_out), epochs, lr, decay, state, noise)
            losses += l
        runs.append((p, np.array(losses)))
    (ref, ref_loss), (off, off_loss) = runs
    losses = np.concatenate([net.train(x, t, m, epochs=e, lr=lr, weight_decay=decay)
                             for e, lr in calls])
    assert np.abs(losses / ref_loss - 1).max() <= 10 * np.abs(off_loss / ref_loss - 1).max() + 2e-6
    err, bound = np.abs(net.get_params() - ref), np.abs(off - ref)
    assert np.median(err) <= 10 * np.median(bound)
    assert np.quantile(err, 0.99) <= 10 * np.quantile(bound, 0.99)
