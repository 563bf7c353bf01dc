"""The predictor's matrix kernels at the edges of their 64-sample tiles: one sample, one
less than a tile, a whole one, one more (the two-launch form), several per block's share."""
import numpy as np
import pytest

from oracle import mlp_oracle as M

pytestmark = pytest.mark.gpu

U = 2.0 ** -24  # f32 rounding


def _bounds(p, x, t):
    """|error| of y and of every gradient of an f32 evaluation: the magnitudes without
    cancellation times the rounding of a chain of up to 1000 operations, plus the whole
    term of a unit so close to 0 that its ReLU may fall on the other side."""
    w1, b1, w2, b2, w3, b3 = p[:1024].reshape(64, 16), p[1024:1088], p[1088:5184].reshape(64, 64), p[5184:5248], \
        p[5248:5312], p[5312]
    a1 = x @ w1.T + b1
    a2 = np.maximum(a1, 0) @ w2.T + b2
    m1 = np.abs(x) @ np.abs(w1).T + np.abs(b1)
    m2 = m1 @ np.abs(w2).T + np.abs(b2)
    my = m2 @ np.abs(w3) + abs(b3)
    md = 2 * (my + np.abs(t)) / len(t)
    d2 = md[:, None] * np.abs(w3)
    d1 = d2 @ np.abs(w2)
    near2, near1 = (np.abs(a2) < 1000 * U * m2), (np.abs(a1) < 1000 * U * m1)
    e2 = d2 * (1000 * U + near2)
    e1 = d1 * (1000 * U + near1) + (d2 * near2) @ np.abs(w2)
    g = np.concatenate([(e1.T @ np.abs(x)).ravel(), e1.sum(0), (e2.T @ m1).ravel(), e2.sum(0), 1000 * U * (md @ m2),
                        [1000 * U * md.sum()]])
    return 1000 * U * my, g


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 63, 64, 65, 127, 128, 129, 1000, 4097, 16500])
def test_tile_edges(n):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from voxelis_amd.predictor import GrowthMLP
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, 16)).astype(np.float32)
    t = rng.uniform(0, 9, n).astype(np.float32)
    net = GrowthMLP(seed=n)
    p = net.p.cpu().numpy().astype(np.float64)
    p[1024:1088] = p[5184:5248] = 0.1  # biases: a padded row of a tile is not zero by itself
    net.p.copy_(torch.from_numpy(p.astype(np.float32)))
    p = net.p.cpu().numpy().astype(np.float64)
    x64, t64 = x.astype(np.float64), t.astype(np.float64)
    g_o, y_o, l_o = M.gradient(p, x64, t64)
    ey, eg = _bounds(p, x64, t64)
    xt, tt = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
    g, y, loss = net.gradient(xt, tt)
    for yy in (y, net.forward(xt)):
        assert np.all(np.abs(yy.cpu().numpy() - y_o) <= ey)
    assert np.all(np.abs(g.cpu().numpy() - g_o) <= eg)
    assert abs(float(loss.item()) - l_o) <= 2 * np.mean(ey * (np.abs(y_o - t64) + ey)) + 1000 * U * l_o
    # a repeat gives the same bits
    g2, y2, loss2 = net.gradient(xt, tt)
    assert torch.equal(g, g2) and torch.equal(y, y2) and torch.equal(loss, loss2)
