"""Steps between two of a cytosol box's own, where they are more than one launch
takes: the effluxes into the box add up over the launches."""
import dataclasses

import numpy as np
import pytest

from casim_amd import abi, workloads
from casim_amd.dyad import DyadHIP
from tests.test_resident import POOL, same
from tests.test_resident2d import state

pytestmark = pytest.mark.gpu


# a launch takes 2048 steps at most: one short of it, a whole one, one more, two and a remainder
@pytest.mark.parametrize("substeps,nx,precision", [(2047, 61, 64), (2048, 41, 32), (2049, 61, 64), (4097, 41, 32),
                                                   (4097, 61, 64)])
def test_long_box_steps(gpu, substeps, nx, precision):
    sp = workloads.coupled_dyads(2, n_ryr=16, extent_nm=120.0,
                                 precision=abi.CASIM_FP32 if precision == 32 else abi.CASIM_FP64)
    sp.channel_types[0].params["kopen0"] *= 1e4
    sp.channel_types[0].params["kclose0"] *= 1e3
    sp.sites = [[(2.0 * (nx // 2 + 4 * i), 2.0 * (30 + 7 * k), 0) for i in range(-2, 3) for k in range(-2, 3)] for _ in range(2)]
    sp = dataclasses.replace(sp, nx=nx, init_channel=[3, 17])
    box = dataclasses.replace(workloads.coupled_box(sp), substeps=substeps)
    dt = sp.meta["dt_ms"] * 50 / substeps
    out = []
    for steps_per_pass in (2, 1):
        d = DyadHIP(sp)
        d.AttachPools(POOL)
        d.AttachCytosolBox(box)
        d.SetStepsPerPass(steps_per_pass)
        d.RecordOpenCounts(500, 40)
        d.InitOpeningAll()
        d.UpdatePools()
        d.SetSplit(False)
        for _ in range(2):
            d.Step(dt, substeps)
        if steps_per_pass == 2:
            assert d.StepPath() == abi.CASIM_STEP_SLABS and d.StepLaunch() == min(substeps, 2048)
        out.append(state(d, sp, None) + [d.GetPools()[0]] + [d.GetCytosolBox(f) for f in range(d.CytosolBoxFields())])
    same(*out)
    assert np.isfinite(out[0][0]).all() and (out[0][-4] != out[0][-4].flat[0]).any()
