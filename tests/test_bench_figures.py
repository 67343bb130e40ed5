"""bench.py prices a leg by what its calls ran, and Step reports what that was."""
import sys

import pytest

from casim_amd import abi, workloads
from casim_amd.dyad import DyadHIP
from tests.conftest import ROOT

LEG = {"sites": 4096, "grid": "81x81x5", "ms_per_step": 0.8, "bytes_per_site_step": 1741072.0, "sweep_launch_ms": 1.6}


@pytest.mark.parametrize("path,per_pass,kernel,label", [
    (abi.CASIM_STEP_SLABS, 2, "k_resident", "state on the chip"),
    (abi.CASIM_STEP_PASSES, 2, "k_sweep2", "two steps per state pass"),
    (abi.CASIM_STEP_PASSES, 1, "k_sweep", "one step per pass")])
def test_leg_figures_follow_the_path(path, per_pass, kernel, label):
    sys.path.insert(0, ROOT)
    import bench
    roofline, sweep, got, whole = bench.plain_leg_figures({**LEG, "step_path": path, "steps_per_launch": per_pass}, abi)
    assert (roofline["kernel"], got) == (kernel, label)
    assert roofline["bound"] == ("fp64" if path == abi.CASIM_STEP_SLABS else "hbm")
    assert sweep["kernel"] == ("k_sweep2" if per_pass == 2 else "k_sweep")
    # a rate of the state's bytes only where every step moves them
    assert whole is None if path == abi.CASIM_STEP_SLABS else abs(whole - 4096 * 1741072.0 / 0.8e-3 / 1e9) < 1e-6 * whole


# small batches stay on the chip at any call length, large ones from about ten steps on
@pytest.mark.gpu
def test_step_reports_its_path(gpu):
    for sites, calls in ((6, ((2, abi.CASIM_STEP_SLABS), (40, abi.CASIM_STEP_SLABS))),
                         (2048, ((2, abi.CASIM_STEP_PASSES), (60, abi.CASIM_STEP_SLABS), (2, abi.CASIM_STEP_PASSES)))):
        sp = workloads.batched_dyads(sites)
        d = DyadHIP(sp)
        d.InitOpeningAll()
        d.Update(*sp.rim_arrays(), sp.jsr_array([1000.0]))
        assert d.StepPath() == 0
        for k, want in calls:
            d.Step(1e-5, k)
            assert (d.StepPath(), d.StepLaunch()) == (want, k), (sites, k)
        d.SetStepsPerPass(1)
        d.Step(1e-5, 60)
        assert d.StepPath() == abi.CASIM_STEP_PASSES
    sp = workloads.coupled_dyads(3, n_ryr=4, extent_nm=60.0)
    d = DyadHIP(sp)
    d.InitOpeningAll()
    d.Update(*sp.rim_arrays(), sp.jsr_array([1000.0]))
    d.Step(1e-6, 1)
    assert d.StepPath() == abi.CASIM_STEP_SITE
