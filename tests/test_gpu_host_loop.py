"""The C++ mirror of simulationLoop (csrc/host/simulate.hpp), by its members."""
import numpy as np
import pytest

import native_lib
from cardioid_amd import hip

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    yield


@pytest.mark.parametrize("n,nstim", [(1, 1), (5, 2), (300, 64), (1030, 1000)])
def test_iStim_holds_the_last_steps_stimulus(n, nstim):
    """Zeroed at a step's start, whatever stood there, and assigned by the
    stimulus that is on: after the loop it is the last step's (elec/
    simulationLoop.cc:186-193).  The pulse is on from step 2 to step 6."""
    steps = np.array([1, 2, 2, 1, 1, 3], np.int32)      # ends after steps 0, 2, 4, 5, 6, 9
    on = [False, True, True, True, True, False]
    out = np.zeros((steps.size, n))
    native_lib.check(native_lib.shim().shim_loop_istim(
        n, nstim, native_lib.C.c_double(0.03), native_lib.C.c_double(0.1),
        native_lib.C.c_double(-7.5), steps.size, hip.ptr(steps, hip.ip),
        native_lib.C.c_double(3.25), hip.ptr(out)))
    for k in range(steps.size):
        want = np.zeros(n)
        want[:nstim] = -7.5 if on[k] else 0.0
        assert np.array_equal(out[k], want), (k, out[k])
