"""The resident form's rules that need no device (csrc/resident_rules.hpp) by
the library's own functions, and the code of its wait."""
import pytest

import native_lib


@pytest.fixture(scope="module")
def shim():
    try:
        return native_lib.shim()
    except Exception as e:      # no library built, no compiler
        pytest.skip(f"no shim: {e}")


def test_only_a_launch_too_large_or_unsupported_falls_back(shim):
    """hip_runtime_api.h: 720 cooperative launch too large, 801 not supported;
    an invalid value, no memory, a sticky fault and the rest are errors."""
    refused = {e for e in range(1200) if shim.shim_resident_refused(e)}
    assert refused == {720, 801}


WAIT = """
#include "engine_resident.hpp"
__global__ void k_wait(cdh::ResidentArgs r, const uint32_t *lk, uint32_t target, int *out)
{
   bool bail = false;
   cdh::resident_wait(r, lk, threadIdx.x, target, bail);
   out[0] = bail;
}
"""


def test_the_bound_of_a_wait_is_no_time_of_day(tmp_path):
    """A clock goes on while a process is held off the chip, for which a wait
    must not fail: it reads none and counts its polls."""
    code = native_lib.device_code(WAIT, tmp_path)
    assert "k_wait" in code and "global_load" in code
    assert "s_memrealtime" not in code and "s_memtime" not in code
