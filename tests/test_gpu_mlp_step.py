"""The training step (rows 16 at a time, gradient in slices of the batch) at
batch sizes around its tiles and slices: the gradient against the CPU
restatement with the same rounding points, and two Adam steps against the
same arithmetic on the step's own gradients."""
import numpy as np
import pytest

import mlp_oracle as MO
from test_gpu_mlp import _ctx, _data, _random_net

pytestmark = pytest.mark.gpu


# one row; a tile's edge; an odd tile filled by a zero one; the first batch
# with two slices; 16 slices; more tiles than workgroups, with a ragged end
@pytest.mark.parametrize("n", [1, 15, 16, 17, 33, 255, 257, 512, 4099, 16411])
def test_gradient_of_any_batch_equals_oracle(n):
    print("mlp gradient of %d rows" % n, flush=True)
    p, scale = _random_net(5)
    X, T, M = _data(n, n)
    C = _ctx()
    try:
        C.set_mlp(p, scale)
        L, g = C.mlp_loss_grad(X, T, M)
        L2, g2 = C.mlp_loss_grad(X, T, M)
    finally:
        C.close()
    assert np.array_equal(g, g2) and abs(L - L2) <= 1e-12 * abs(L)
    Lo, go = MO.loss_grad(p, MO.standardise(X, scale), MO.scale_targets(T, scale), M, exact=False)
    # the bounds of the 2048-row gradient: a BF16 rounding that falls the
    # other way moves an activation by 2^-8
    assert abs(L - Lo) / Lo < 1e-3
    for (ow, ob), (k, m) in zip(MO.OFFS, MO.LAYERS):
        for a, b in ((ow, ow + m * k), (ob, ob + m)):
            assert np.linalg.norm(g[a:b] - go[a:b]) / np.linalg.norm(go[a:b]) < 1e-2, (a, b)
    assert np.all(g[MO.OFFS[0][0]:MO.OFFS[0][1]].reshape(128, 96)[:, 72:] == 0)


@pytest.mark.parametrize("n", [17, 600])
def test_two_steps_are_adam_on_the_gradients(n):
    """The second step's gradient is taken at the parameters of the first, so
    it sees both BF16 copies refreshed.  Both sides start each step from the
    device's parameters: one off by an ulp can round to another BF16 weight."""
    print("mlp steps of %d rows" % n, flush=True)
    lr = 1e-3
    p, scale = _random_net(6)
    X, T, M = _data(7, n)
    order = np.arange(n, dtype=np.int32)
    C = _ctx()
    try:
        at, want = p.astype(np.float32), []
        m, v = np.zeros_like(at), np.zeros_like(at)
        got = []
        for t in (1, 2):
            C.set_mlp(at, scale)
            g = C.mlp_loss_grad(X, T, M)[1].astype(np.float32)
            m = np.float32(0.9) * m + np.float32(0.1) * g
            v = np.float32(0.999) * v + np.float32(0.001) * g * g
            want.append(at - np.float32(lr) * (m / np.float32(1 - 0.9 ** t)) /
                        (np.sqrt(v / np.float32(1 - 0.999 ** t)) + np.float32(1e-8)))
            C.set_mlp(p, scale)
            C.mlp_train(X, T, M, np.tile(order, t), n, lr)
            at = C.get_mlp()[0]
            got.append(at)
    finally:
        C.close()
    # an update is lr times a ratio of order one; both sides take it in FP32
    for a, b in zip(got, want):
        assert np.max(np.abs(a - b)) < 1e-3 * lr + 2.0 ** -23 * np.max(np.abs(b))
