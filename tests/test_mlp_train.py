"""Training steps of every member in two launches against a layer and a member
at a time, bit for bit: every product, sum and update is formed by the same
operations in the same order."""
import numpy as np
import pytest

from casim_amd.mlp import MLP

pytestmark = pytest.mark.gpu


def trained(fused, n_in, width, depth, members, rows, batch, epochs):
    g = np.random.default_rng(rows)
    x = g.standard_normal((rows, n_in)).astype(np.float32)
    y = (np.sin(x).sum(1) + 3.0).astype(np.float32)
    m = MLP(n_in, width=width, depth=depth, members=members, seed=5)
    m.fit_normalization(x, y)
    m.set_data(x, y)
    m.set_fused(fused)
    loss = [m.train(1, batch=batch, lr=1e-3, seed=2), m.train(epochs, batch=batch, lr=3e-3, seed=9)]
    return loss, [m.params(e) for e in range(members)], m.predict(x[:70])


# one feature and the widest, one hidden layer and the most, one member and the
# most, batches of one row, around a tile of 32, not a multiple of it, and the
# whole set; rows left over at the end of an epoch
@pytest.mark.parametrize("n_in,width,depth,members,rows,batch,epochs", [
    (57, 256, 4, 5, 1500, 400, 2), (1, 64, 1, 1, 70, 31, 3), (256, 192, 7, 8, 130, 33, 2), (33, 64, 2, 3, 40, 32, 2),
    (12, 128, 3, 2, 9, 1, 1), (65, 256, 2, 4, 77, 500, 3)])
def test_two_launch_steps_equal_the_layer_path(gpu, n_in, width, depth, members, rows, batch, epochs):
    shape = (n_in, width, depth, members, rows, batch, epochs)
    (la, pa, oa), (lb, pb, ob) = trained(True, *shape), trained(False, *shape)
    assert np.isfinite(pa).all()
    np.testing.assert_array_equal(pa, pb)
    np.testing.assert_array_equal(la, lb)
    for u, v in zip(oa, ob):
        np.testing.assert_array_equal(u, v)
