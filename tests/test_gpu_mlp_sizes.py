"""The fused training kernels at the batches where they can go wrong: one row,
one row less and more than a 32-row tile, one tile a block (8,192 rows) and the
blocks' second tile; the rows of a training step are the drawn samples.
  gradient vs the FP64 oracle: relative L2 <= 1e-5 (FP32 sums of at most 64
    products in five layers, 2^-24 * sqrt(64) * 5 ~ 2.4e-6, times 4), loss
    rel <= 1e-6.  Small batches of O(1) residuals: no cancellation in the sums.
  first loss of a training step vs the oracle over the rows that Philox draws:
    rel <= 1e-5."""
import numpy as np
import pytest

import o_mlp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 2, 31, 32, 33, 511, 8192, 8193, 16415])
def test_gradient_by_batch(pkg, rows):
    s = pkg.Solver(precision="fp32s")
    s.mlp_init(21)
    p, _, _ = s.mlp_get_params()
    rng = np.random.default_rng(rows)
    X = rng.uniform(-1, 1, (rows, 12)).astype(np.float32)
    y = rng.normal(0, 1, rows).astype(np.float32)
    loss, g = s.mlp_loss_grad(X, y)
    loss_o, g_o = o_mlp.loss_and_grad(p.astype(np.float64), X.astype(np.float64),
                                      y.astype(np.float64))
    e = float(np.linalg.norm(g - g_o) / np.linalg.norm(g_o))
    print(f"{rows} rows: gradient relL2 {e:.2e}, loss {loss:.6e} vs {loss_o:.6e}")
    assert e <= 1e-5 and abs(loss - loss_o) <= 1e-6 * loss_o
    ref, _ = o_mlp.forward(p.astype(np.float64), X.astype(np.float64))
    assert np.abs(s.mlp_forward(X, mfma=False) - ref).max() <= 1e-5 * (1 + np.abs(ref).max())
    # a smaller batch after a larger one, on the same workspace
    if rows > 40:
        k = rows // 3
        _, g = s.mlp_loss_grad(X[:k], y[:k])
        _, g_o = o_mlp.loss_and_grad(p.astype(np.float64), X[:k].astype(np.float64),
                                     y[:k].astype(np.float64))
        assert np.linalg.norm(g - g_o) <= 1e-5 * np.linalg.norm(g_o)


@pytest.mark.parametrize("batch", [5, 32, 1000, 8229])
def test_training_step_takes_the_drawn_rows(pkg, orc, batch):
    s = pkg.Solver(precision="fp32s", nu=0.003, alpha_tol=1e-10)
    s.define_level(0, (20, 18, 17))
    s.init_tgv(0, 0.05, 1e-3, 3)
    s.step(0, 3)
    s.mlp_reserve(2 * 20 * 18 * 17)
    n = [s.mlp_collect(0, 1) for _ in range(2)][-1]
    s.mlp_init(8)
    p, _, _ = s.mlp_get_params()
    seed = (5 << 32) + 77
    first, last = s.mlp_train(1, batch, 2e-3, seed)
    assert first == last
    X, y = s.mlp_samples(n)  # the targets are normalised by now
    assert abs(y.mean()) < 1e-3 and abs(y.std() - 1) < 1e-3
    at = []
    for r in range(batch):
        c = orc.philox((r, 0, 0, 0x6d6c70), (seed & 0xffffffff, seed >> 32))
        at.append(((int(c[0]) << 32) | int(c[1])) % n)
    want, g = o_mlp.loss_and_grad(p.astype(np.float64), X[at].astype(np.float64),
                                  y[at].astype(np.float64))
    assert abs(first - want) <= 1e-5 * want
    # Adam's first step moves each parameter by lr g / (|g| + eps), eps 1e-8
    q, _, _ = s.mlp_get_params()
    clear = np.abs(g) > 1e-4
    assert clear.sum() > 100
    assert np.abs((p - q)[clear] - 2e-3 * np.sign(g[clear])).max() <= 1e-5
