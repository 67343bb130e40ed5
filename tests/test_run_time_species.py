"""Two steps per pass against one with species that have no compiled layout, bit
for bit, over the nodes of a plane that a thread takes."""
import dataclasses

import numpy as np
import pytest

from casim_amd import abi, workloads
from casim_amd.config import Buffer
from casim_amd.dyad import DyadHIP
from tests.test_resident import POOL, same
from tests.test_resident2d import state

pytestmark = pytest.mark.gpu


# one, two and four nodes per thread (the last one takes one step per pass)
@pytest.mark.parametrize("nx,ny,nz,precision,per_pass", [
    (61, 200, 1, 64, 2), (61, 380, 1, 64, 2), (41, 600, 1, 32, 1), (41, 250, 1, 32, 2), (41, 50, 5, 64, 2), (41, 81, 5, 32, 2),
    (31, 121, 5, 32, 1)])
def test_pairs_equal_single_steps(gpu, nx, ny, nz, precision, per_pass):
    p = abi.CASIM_FP32 if precision == 32 else abi.CASIM_FP64
    sp = workloads.coupled_dyads(3, n_ryr=16, precision=p) if nz == 1 else workloads.batched_dyads(3, precision=p)
    sp.channel_types[0].params["kopen0"] *= 1e5
    sp.channel_types[0].params["kclose0"] *= 1e4
    sp.buffers = sp.buffers + [Buffer("Z", 50.0, {sp.ions[0].name: (0.0, 0.05, 0.3)})]
    sp.sites = [[(sp.dx * (nx // 2 + 3 * i), sp.dy * (ny // 2 + 4 * k), 0) for i in range(-2, 3) for k in range(-2, 3)]
                for _ in range(3)]
    sp = dataclasses.replace(sp, nx=nx, ny=ny, nz=nz, init_channel=[0, 7, 24])
    if nz > 1:
        sp = dataclasses.replace(sp, z=4.0 * (nz - 1))
    out = []
    for steps in (2, 1):
        d = DyadHIP(sp)
        d.AttachPools(POOL)
        d.SetStepsPerPass(steps)
        d.RecordOpenCounts(5, 40)
        assert d.StepsPerPass() == (per_pass if steps == 2 else 1)
        d.InitOpeningAll()
        d.UpdatePools(*sp.rim_arrays())
        for k in (50, 7, 80):
            d.Step(sp.meta["dt_ms"], k)
        assert d.StepPath() == abi.CASIM_STEP_PASSES
        out.append(state(d, sp, None))
    same(*out)
    assert np.isfinite(out[0][0]).all() and (out[0][0] != out[0][0].flat[0]).any()
