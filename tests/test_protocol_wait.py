"""The protocol calls return when their device work is done."""
import ctypes as C

import pytest

from casim_amd import workloads
from casim_amd.dyad import DyadHIP

pytestmark = pytest.mark.gpu


# small batches send the update's inputs in one pinned copy, large ones as they are
@pytest.mark.parametrize("sites", [200, 1500])
def test_stream_is_idle_after_each_protocol_call(gpu, sites):
    sp = workloads.batched_dyads(sites)
    d = DyadHIP(sp)
    d.InitOpeningAll()
    rim, jsr = sp.rim_arrays(), sp.jsr_array([1000.0])
    hip = C.CDLL("libamdhip64.so")
    stream = C.c_void_p(d.stream())
    for _ in range(3):
        for call in (lambda: d.Update(*rim, jsr), lambda: d.RunRD(1e-5), lambda: d.RunMC(1e-5)):
            call()
            assert hip.hipStreamQuery(stream) == 0  # 600: work still runs
