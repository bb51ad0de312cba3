"""The cost model's kernels at the edges of their 16 x 16 tiles, of the k steps
of 32 and of the vector loads (widths that are no multiple of 4), and one
training step against Adam applied to the gradients. Gradients: 2e-2 of a
block's largest magnitude against the FP32 reference with the same bfloat16
operands, for the order of summation. The step: both sides use the same FP32
gradients, so they differ by the rounding of about ten operations, 1e-6 of the
step, and of one subtraction, 1.2e-7 of the parameter (an ulp)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def blocks(in_dim, hidden):
    sizes = [in_dim * hidden, hidden, hidden * hidden, hidden, hidden, 1]
    ends = np.cumsum(sizes)
    return [slice(e - n, e) for e, n in zip(ends, sizes)]


@pytest.mark.parametrize("in_dim,hidden,batch", [(1, 1, 1), (5, 17, 16), (33, 30, 31), (96, 64, 257), (64, 256, 770),
                                                 (31, 16, 2100)])
def test_gradients_and_one_step(gat, gpu, in_dim, hidden, batch):
    from graphautotune_amd.tuning import mlp
    m = mlp.MLPCostModel(in_dim, hidden, seed=7)
    rng = np.random.default_rng(in_dim)
    X = rng.normal(size=(batch, in_dim)).astype(np.float32)
    t = rng.normal(size=batch).astype(np.float32)
    p0 = m.params()
    g, loss = m.gradients(X, t)
    want, want_loss = mlp.reference_gradients(p0, X.astype(np.float64), t.astype(np.float64), in_dim, hidden)
    assert abs(loss - want_loss) <= 2e-3 * max(1.0, abs(want_loss))
    for s in blocks(in_dim, hidden):
        assert np.abs(g[s] - want[s]).max() <= 2e-2 * max(np.abs(want[s]).max(), 1e-12), s
    lr = 2e-3
    assert m.train_raw(X, t, 1, lr) == pytest.approx(loss, rel=1e-6)
    g64 = g.astype(np.float64)
    step = lr * g64 / (np.abs(g64) + 1e-8)  # first step: m / c1 = g, v / c2 = g^2
    p1 = m.params()
    tol = 1e-5 * lr + 2.4e-7 * np.abs(p0)
    assert (np.abs(p1 - (p0 - step)) <= tol).all(), np.abs(p1 - (p0 - step)).max()
