"""A step whose workgroups may not wait for each other gives up right away: every
kernel ends as usual, every call says that the state is invalid, and no later
launch of the handle waits for workgroups that have left."""
import time

import numpy as np
import pytest

from casim_amd import abi, workloads
from casim_amd.dyad import DyadHIP
from tests.test_resident import POOL, same, spec, start

pytestmark = pytest.mark.gpu

GAVE_UP = pytest.raises(abi.CasimError, match="gave up")


def boxed():
    sp = workloads.coupled_dyads(3, n_ryr=16, extent_nm=120.0)
    d = DyadHIP(sp)
    d.AttachPools(POOL)
    d.AttachCytosolBox(workloads.coupled_box(sp))
    d.InitOpeningAll()
    d.UpdatePools()
    return sp, d


def plain():
    sp = spec(4, 81, 81, 5, abi.CASIM_FP64)  # 16 workgroups to a site
    return sp, start(sp, False, 2)


def give_up(d, dt, k=500):
    d.SetWaitLimit(0.0)
    d.Step(dt, k)
    assert d.StepPath() == abi.CASIM_STEP_SLABS
    d.SetWaitLimit(20.0)


@pytest.mark.parametrize("box", [False, True])
def test_every_call_reports_it(gpu, box):
    sp, d = boxed() if box else plain()
    dt = sp.meta["dt_ms"]
    give_up(d, dt)
    calls = [d.Synchronize, lambda: d.Step(dt, 100), lambda: d.StepProfiled(dt, 100), lambda: d.GetField(0),
             d.GetConcentrations, d.GetChannelsStates, d.GetRngStates, d.GetIonsNearChannels, d.GetEffluxes,
             d.GetTotalSRCurrent, d.GetReleaseStats, d.InitOpeningAll, lambda: d.RunMC(dt),
             lambda: d.SetField(0, np.ones(sp.n_sites * sp.nodes_per_site()))]
    if box:
        calls += [lambda: d.GetCytosolBox(0), lambda: d.SetCytosolBox(0, np.ones(3 * 51 ** 3)), d.UpdatePools, d.GetPools]
    else:
        calls += [lambda: d.RunRD(dt), lambda: d.Update(*sp.rim_arrays(), sp.jsr_array([1000.0])), d.GetOpenCounts]
    for c in calls:
        with GAVE_UP:
            c()
    d.close()


def test_later_launches_do_not_wait(gpu):
    """The second call is most likely enqueued before the first one has given up;
    its workgroups stand at different steps."""
    sp, d = plain()
    t = time.perf_counter()
    give_up(d, 1e-5)
    with GAVE_UP:
        d.Step(1e-5, 500)
        d.Synchronize()
    assert time.perf_counter() - t < 5.0  # a wait takes 20 s


@pytest.mark.parametrize("box", [False, True])
def test_reset_makes_the_handle_usable_again(gpu, box):
    out = []
    for fail in (True, False):
        sp, d = boxed() if box else plain()
        dt = sp.meta["dt_ms"]
        if fail:
            for _ in range(2):  # the second time after a whole run
                give_up(d, dt)
                with GAVE_UP:
                    d.Synchronize()
                d.Reset()
                d.InitOpeningAll()
                d.UpdatePools() if box else d.Update(*sp.rim_arrays(), sp.jsr_array([1000.0]))
                d.Step(dt, 100)
                d.Synchronize()
            d.Reset()
            d.InitOpeningAll()
            d.UpdatePools() if box else d.Update(*sp.rim_arrays(), sp.jsr_array([1000.0]))
        for k in (50, 100, 350):
            d.Step(dt, k)
        out.append([d.GetField(f) for f in range(sp.n_ions + sp.n_bound)] +
                   [d.GetChannelsStates(), d.GetRngStates(), d.GetTotalSRCurrent(), d.GetReleaseStats()] +
                   ([d.GetCytosolBox(f) for f in range(d.CytosolBoxFields())] if box else []))
    same(*out)


def test_limit_is_checked(gpu):
    sp, d = plain()
    for bad in (-1.0, 3601.0, float("nan")):
        with pytest.raises(abi.CasimError, match="limit"):
            d.SetWaitLimit(bad)
    d.SetWaitLimit(0.5)
    d.Step(1e-5, 500)
    d.Synchronize()
