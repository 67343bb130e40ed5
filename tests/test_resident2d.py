"""Steps of 2D sites with the state in LDS (resident2d.hip) against one state
pass per step, bit for bit: the operations and their order are the same."""
import dataclasses
import os

import numpy as np
import pytest

from casim_amd import abi, config, workloads
from casim_amd.dyad import DyadHIP
from tests.conftest import GOLDEN
from tests.test_resident import POOL, same

pytestmark = pytest.mark.gpu


def spec(kind, sites, nx, ny, precision):
    """One ion on the coupled configuration's 2D cleft, or the reference's test
    input with its two ions; clusters of 1 to 127 RyRs around the centre, two
    channels on a node, gating fast enough to toggle within a call."""
    pools = None
    if kind == "one_ion" or kind == "jsr":
        sp = workloads.coupled_dyads(sites, n_ryr=4, extent_nm=80.0)
        sp.channel_types[0].params["kopen0"] *= 1e5
        pools = POOL if kind == "jsr" else None
    else:
        sp, j = config.load_json(os.path.join(GOLDEN, "test_input_Parameters.json"), n_sites=sites)
        if kind == "cytosol":
            pools = config.pools_from_json(j, sp)
    cells = [(sp.dx * (nx // 2 + i), sp.dy * (ny // 2 + k), 0) for i in range(-5, 6) for k in range(-6, 7)]
    if min(nx, ny) < 16:
        cells = [(sp.dx * (nx // 2 + i), sp.dy * (ny // 2 + k), 0) for i in range(-1, 2) for k in range(-1, 2)]
    cells.sort(key=lambda c: ((c[0] - sp.dx * (nx // 2)) ** 2 + (c[1] - sp.dy * (ny // 2)) ** 2, c))
    sizes = (127, 64, 1, 65, 20)
    site = [cells[:min(sizes[s % 5], len(cells))] for s in range(sites)]
    site = [c + [c[0]] if len(c) < 100 else c for c in site]
    return dataclasses.replace(sp, nx=nx, ny=ny, sites=site, precision=precision, init_channel=[0] * sites), pools


def start(sp, pools, steps_per_pass):
    d = DyadHIP(sp)
    if pools is not None:
        d.AttachPools(pools)
    d.SetStepsPerPass(steps_per_pass)
    d.RecordOpenCounts(5, 40)
    d.InitOpeningAll()
    rim = sp.rim_arrays()
    if pools is not None:
        d.UpdatePools(*rim)
    else:
        d.Update(*rim, sp.jsr_array([1000.0] * sp.n_ions))
    return d


def state(d, sp, pools):
    out = [d.GetField(f) for f in range(sp.n_ions + sp.n_bound)]
    out += [d.GetChannelsStates(), d.GetRngStates(), d.GetIonsNearChannels(), d.GetTotalSRCurrent(), d.GetEffluxes(),
            d.GetReleaseStats(), d.GetOpenCounts()]
    return out + (list(d.GetPools()) if pools is not None else [])


# the smallest grid, a node wave full and one node over, the most nodes, more
# sites than CUs, and (last) a grid that does not fit and takes the sweeps
@pytest.mark.parametrize("kind,sites,nx,ny,precision", [
    ("cytosol", 3, 31, 41, 64), ("cytosol", 300, 21, 20, 64), ("cytosol", 2, 31, 41, 32), ("two_ions", 5, 5, 9, 64),
    ("two_ions", 2, 34, 58, 64), ("jsr", 6, 18, 10, 64), ("jsr", 2, 45, 43, 32), ("one_ion", 2, 10, 18, 64),
    ("one_ion", 3, 40, 47, 64), ("one_ion", 2, 45, 46, 64)])
def test_equals_one_step_per_pass(gpu, kind, sites, nx, ny, precision):
    sp, pools = spec(kind, sites, nx, ny, abi.CASIM_FP32 if precision == 32 else abi.CASIM_FP64)
    dt = 1e-6
    a, b = start(sp, pools, 2), start(sp, pools, 1)
    for k in (50, 1, 2, 2100):  # the last one takes more than one launch
        a.Step(dt, k)
        b.Step(dt, k)
    sa = state(a, sp, pools)
    same(sa, state(b, sp, pools))
    assert np.isfinite(sa[0]).all()
    # other step forms go on from it, and it goes on from them and from a state set by hand
    a.SetStepsPerPass(1)
    for d in (a, b):
        d.Step(dt, 3)
        d.SetChannelsStates(1 - d.GetChannelsStates())
        d.Step(dt, 1)
    a.SetStepsPerPass(2)
    for d in (a, b):
        d.Step(dt, 41)
    same(state(a, sp, pools), state(b, sp, pools))


# grids that take several workgroups per site, with and without a cytosol box:
# halves of a slab that differ and that do not, rows of one wave and of three,
# doubled rows, more sites than fit at once; the last one takes the sweeps
@pytest.mark.parametrize("sites,nx,ny,precision,box", [
    (3, 61, 61, 64, True), (45, 201, 201, 64, True), (2, 63, 101, 64, False), (9, 41, 61, 32, True), (4, 72, 206, 32, False),
    (2, 68, 50, 64, True), (2, 60, 207, 64, False)])
def test_wide_grid_equals_one_step_per_pass(gpu, sites, nx, ny, precision, box):
    sp = workloads.coupled_dyads(sites, n_ryr=16, extent_nm=2.0 * (min(nx, ny) - 1),
                                 precision=abi.CASIM_FP32 if precision == 32 else abi.CASIM_FP64)
    sp.channel_types[0].params["kopen0"] *= 1e5
    sp.channel_types[0].params["kclose0"] *= 1e4
    c = min(nx, ny) // 2
    sp.sites = [[(2.0 * (nx // 2 + i * (c // 4)), 2.0 * (ny // 2 + k * (c // 4)), 0) for i in range(-2, 3) for k in range(-2, 3)]
                for _ in range(sites)]
    sp = dataclasses.replace(sp, nx=nx, ny=ny, init_channel=[s % 25 for s in range(sites)])
    devs = []
    for steps_per_pass in (2, 1):
        d = DyadHIP(sp)
        d.AttachPools(POOL)
        if box:
            d.AttachCytosolBox(workloads.coupled_box(sp))
        d.SetStepsPerPass(steps_per_pass)
        d.RecordOpenCounts(5, 40)
        d.InitOpeningAll()
        d.UpdatePools(*(() if box else sp.rim_arrays()))
        for k in (50, 150):
            d.Step(sp.meta["dt_ms"], k)
        out = state(d, sp, None) + [d.GetPools()[0]]
        devs.append(out + [d.GetCytosolBox(f) for f in range(4)] if box else out)
    same(*devs)
    assert np.isfinite(devs[0][0]).all() and (devs[0][0] != devs[0][0].flat[0]).any()
