"""Steps with the state on the chip (resident.hip) against one state pass per
step, bit for bit: both evaluate node_update's operations in its order, form
the same currents and draw the same numbers, so nothing may differ."""
import dataclasses

import numpy as np
import pytest

from casim_amd import abi, workloads
from casim_amd.config import PoolSpec
from casim_amd.dyad import DyadHIP

pytestmark = pytest.mark.gpu

POOL = PoolSpec(jsr_constant=False, jsr_cq_total=10000.0, jsr_volume=2e5, jsr_c0=[1000.0], jsr_cq_sites=[1.0],
                jsr_k_cq=[800.0], jsr_tau_refill=[100.0], nsr_c=[1000.0])


def spec(sites, nx, ny, nz, precision):
    """Clusters of 1 to 127 RyRs (two channel chunks), gating fast enough to
    toggle within a call; two channels of the first sites share a node."""
    sp = workloads.batched_dyads(sites, geometry_seed=nx + ny, precision=precision)
    sp.channel_types[0].params["kopen0"] *= 1e5
    sp.channel_types[0].params["kclose0"] *= 1e4
    cx, cy, pitch = 2.0 * (nx - 1), 2.0 * (ny - 1), 4.0 * ((min(nx, ny) - 8) // 12)
    cells = sorted(((cx + pitch * (i - 5.5), cy + pitch * (j - 5.5), 0) for i in range(12) for j in range(12)),
                   key=lambda p: ((p[0] - cx) ** 2 + (p[1] - cy) ** 2, p[0], p[1]))
    sp.sites = [cells[:(127, 64, 1, 65, 63, 20)[s % 6]] for s in range(sites)]
    sp.sites = [c + [c[0]] if s < 9 and len(c) < 100 else c for s, c in enumerate(sp.sites)]
    return dataclasses.replace(sp, nx=nx, ny=ny, nz=nz, z=4.0 * (nz - 1))


def start(sp, pool, steps_per_pass):
    d = DyadHIP(sp)
    if pool:
        d.AttachPools(POOL)
    d.SetStepsPerPass(steps_per_pass)
    d.RecordOpenCounts(5, 40)
    d.InitOpeningAll()
    ri, rb = sp.rim_arrays()
    if pool:
        d.UpdatePools(ri, rb)
    else:
        d.Update(ri, rb, sp.jsr_array([1000.0]))
    return d


def state(d, sp, pool):
    out = [d.GetField(f) for f in range(sp.n_ions + sp.n_bound)]
    out += [d.GetChannelsStates(), d.GetRngStates(), d.GetIonsNearChannels(), d.GetTotalSRCurrent(), d.GetEffluxes(),
            d.GetReleaseStats(), d.GetOpenCounts()]
    return out + ([d.GetPools()[0]] if pool else [])


def same(a, b):
    for i, (x, y) in enumerate(zip(a, b)):
        assert np.array_equal(x, y), i


# slabs per site 1 to 16, the middle planes of a slab held once and twice, the
# last node wave full, nearly empty and absent, more sites than fit at once,
# planes of more than seven node waves, and (the last one) planes that do not
# fit and take the sweeps
@pytest.mark.parametrize("sites,nx,ny,nz,precision,pool", [
    (1, 81, 81, 5, 64, False), (7, 48, 88, 5, 64, True), (3, 59, 61, 2, 64, False), (40, 81, 79, 5, 64, False),
    (40, 81, 88, 5, 64, True), (90, 73, 64, 4, 64, True), (30, 52, 52, 5, 64, False), (2, 95, 77, 5, 32, True), (150, 81, 81, 5, 32, False),
    (70, 62, 49, 4, 32, False), (20, 87, 51, 5, 32, True), (3, 60, 89, 5, 64, False), (34, 85, 96, 6, 64, True),
    (70, 83, 95, 6, 32, False), (5, 49, 128, 4, 32, True), (3, 60, 130, 3, 64, False)])
def test_equals_one_step_per_pass(gpu, sites, nx, ny, nz, precision, pool):
    sp = spec(sites, nx, ny, nz, abi.CASIM_FP32 if precision == 32 else abi.CASIM_FP64)
    a, b = start(sp, pool, 2), start(sp, pool, 1)
    for k in (50, 2, 1, 33) + ((2100,) if sites < 4 else ()):  # the longest takes two launches
        a.Step(1e-5, k)
        b.Step(1e-5, k)
    sa = state(a, sp, pool)
    same(sa, state(b, sp, pool))
    assert np.isfinite(sa[0]).all() and (sa[sp.n_ions + sp.n_bound] == 1).any()
    # other step forms go on from it, and it goes on from them and from a state set by hand
    a.SetStepsPerPass(1)
    for d in (a, b):
        d.Step(1e-5, 3)
        d.SetChannelsStates(1 - d.GetChannelsStates())
        d.Step(1e-5, 1)
    a.SetStepsPerPass(2)
    for d in (a, b):
        d.Step(1e-5, 41)
    same(state(a, sp, pool), state(b, sp, pool))


# a call too short to pay takes the sweeps and keeps nothing; longer and short
# ones after it, in either order
def test_short_calls_before_and_between_long_ones(gpu):
    sp = spec(600, 52, 50, 5, abi.CASIM_FP64)
    a, b = start(sp, False, 2), start(sp, False, 1)
    for k in (2, 2, 60, 2, 60):
        a.Step(1e-5, k)
        b.Step(1e-5, k)
    same(state(a, sp, False), state(b, sp, False))


def test_two_handles_step_beside_each_other(gpu):
    """Launches of two handles share the chip: more workgroups than fit."""
    sp = spec(60, 81, 81, 5, abi.CASIM_FP64)
    one = start(sp, False, 1)
    one.Step(1e-5, 120)
    want = state(one, sp, False)
    devs = [start(sp, False, 2) for _ in range(3)]
    for _ in range(3):
        for d in devs:
            d.Step(1e-5, 40)
    for d in devs:
        same(state(d, sp, False), want)
