"""Batches of casim_mlp_predict that take several pinned slots."""

import numpy as np
import pytest

from casim_amd.mlp import MLP

pytestmark = pytest.mark.gpu


# slots of 16384 rows, and of 4096 where 1500 features make a row wide: one row
# short of a slot, a whole one, one row more and a third slot that reuses the first.
# Each piece runs the same launches alone, so the outputs are the same bits.
@pytest.mark.parametrize("n_in,slot", [(12, 16384), (1500, 4096)])
@pytest.mark.parametrize("extra", [-1, 0, 1])
@pytest.mark.parametrize("whole", [1, 2])
def test_slots_equal_their_pieces(gpu, n_in, slot, extra, whole):
    rows = whole * slot + extra
    x = np.random.default_rng(rows).standard_normal((rows, n_in)).astype(np.float32)
    m = MLP(n_in, width=64, depth=2, members=2, seed=3)
    got = m.predict(x)
    parts = [m.predict(x[r:r + slot]) for r in range(0, rows, slot)]
    for k, g in enumerate(got):
        assert np.isfinite(g).all()
        np.testing.assert_array_equal(g, np.concatenate([p[k] for p in parts], axis=-1))
