"""Sites without channels keep their streams in the kernels that hold the state
on the chip, as in one state pass per step: no draw is taken."""
import numpy as np
import pytest

from casim_amd import abi
from casim_amd.dyad import DyadHIP
from tests import test_resident, test_resident2d
from tests.test_resident import POOL, same

pytestmark = pytest.mark.gpu


def started(sp, pools, steps_per_pass):
    d = DyadHIP(sp)
    if pools is not None:
        d.AttachPools(pools)
    d.SetStepsPerPass(steps_per_pass)
    d.RecordOpenCounts(5, 40)
    for s, cells in enumerate(sp.sites):
        if cells:
            d.InitOpening(s, sp.init_channel[s])
    rim = sp.rim_arrays()
    if pools is not None:
        d.UpdatePools(*rim)
    else:
        d.Update(*rim, sp.jsr_array([1000.0] * sp.n_ions))
    return d


def everything(d, sp, pools):
    out = [d.GetField(f) for f in range(sp.n_ions + sp.n_bound)]
    out += [d.GetChannelsStates(), d.GetRngStates(), d.GetIonsNearChannels(), d.GetTotalSRCurrent(), d.GetEffluxes(),
            d.GetReleaseStats(), d.GetOpenCounts()]
    return out + (list(d.GetPools()) if pools is not None else [])


# a slab and 16 slabs to a site in 3D, two slabs to a workgroup in 2D, a workgroup
# per site with and without compartments; every third site empty, then all of them
@pytest.mark.parametrize("every", [3, 1])
@pytest.mark.parametrize("kind,sites,nx,ny", [("3d", 4, 81, 81), ("3d jsr", 300, 22, 40), ("one_ion", 3, 60, 71),
                                              ("one_ion", 4, 18, 20), ("cytosol", 7, 31, 41)])
def test_streams_of_empty_sites_stay(gpu, kind, sites, nx, ny, every):
    if kind.startswith("3d"):
        sp, pools = test_resident.spec(sites, nx, ny, 5, abi.CASIM_FP64), POOL if kind == "3d jsr" else None
        dt = 1e-5
    else:
        sp, pools = test_resident2d.spec(kind, sites, nx, ny, abi.CASIM_FP64)
        dt = 1e-6
    sp.sites = [[] if s % every == 0 else c for s, c in enumerate(sp.sites)]
    sp.init_channel = [0] * sites
    devs = [started(sp, pools, steps_per_pass) for steps_per_pass in (2, 1)]
    begin = devs[0].GetRngStates()
    for d in devs:
        for k in (40, 3, 60):
            d.Step(dt, k)
    empty = [s for s in range(sites) if not sp.sites[s]]
    np.testing.assert_array_equal(devs[0].GetRngStates()[empty], begin[empty])
    same(*[everything(d, sp, pools) for d in devs])
    devs[0].SetRngStates(devs[0].GetRngStates())
