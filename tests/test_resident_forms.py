"""Batches between those of test_resident.py, so that every compiled form of
k_resident is compared with one state pass per step."""
import pytest

from casim_amd import abi
from tests.test_resident import same, spec, start, state

pytestmark = pytest.mark.gpu


# FP32: slabs of 5, 10 and 20 planes of up to 440 nodes and of up to 576; FP64: of 5 and 10 planes of both, 20 of 409 to 440
@pytest.mark.parametrize("sites,nx,ny,nz,precision,pool", [
    (12, 81, 81, 5, 32, False), (25, 81, 81, 5, 32, True), (60, 81, 81, 5, 32, False), (3, 60, 96, 6, 32, True),
    (25, 81, 95, 6, 32, False), (60, 81, 96, 6, 32, False), (12, 81, 81, 5, 64, True), (25, 81, 81, 5, 64, False),
    (3, 70, 96, 6, 64, False), (25, 81, 95, 6, 64, True), (60, 81, 83, 5, 64, False)])
def test_equals_one_step_per_pass(gpu, sites, nx, ny, nz, precision, pool):
    sp = spec(sites, nx, ny, nz, abi.CASIM_FP32 if precision == 32 else abi.CASIM_FP64)
    a, b = start(sp, pool, 2), start(sp, pool, 1)
    for k in (60, 45):
        a.Step(1e-5, k)
        b.Step(1e-5, k)
    assert (a.StepPath(), b.StepPath()) == (abi.CASIM_STEP_SLABS, abi.CASIM_STEP_PASSES)
    same(state(a, sp, pool), state(b, sp, pool))
